// Host side of liblact_hip.so: validates a program, lays out the caller's buffers and enqueues the
// kernels of the forward and backward passes on the caller's stream.  No allocation, no
// synchronisation, no torch types.
#include "../../include/lact_hip.h"

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <climits>
#include <cstring>
#include <string>
#include <vector>
#include <mutex>
#include <memory>

#include <type_traits>

#include "gemm_dma_kernels.h"
#include "ns_fused.h"
#include "ns_local.h"
#include "gemm_persist.h"
#include "gemm_wide.h"
#include "gemm_kernels.h"
#include "state_kernels.h"
#include "layer_kernels.h"
#include "window_attention.h"
#include "small_heads.h"
#include "plan.h"

using namespace lact;

namespace {

// ---- optional per-launch timing (HIP events on the caller's stream) ---------------------------------
struct ProfRec {
  const char* kernel;
  const char* site;
  double flops;
  hipStream_t stream;
  hipEvent_t e0, e1;
};
struct Profiler {
  bool on = false;
  std::vector<ProfRec> recs;
  std::vector<hipEvent_t> pool;
  hipEvent_t get() {
    if (!pool.empty()) {
      hipEvent_t e = pool.back();
      pool.pop_back();
      return e;
    }
    hipEvent_t e;
    (void)hipEventCreate(&e);
    return e;
  }
  void clear() {
    for (auto& r : recs) {
      pool.push_back(r.e0);
      pool.push_back(r.e1);
    }
    recs.clear();
  }
};
Profiler g_prof;
struct ProfScope {
  hipStream_t s;
  hipEvent_t e1 = nullptr;
  ProfScope(const char* kernel, const char* site, double flops, hipStream_t st) : s(st) {
    if (!g_prof.on) return;
    ProfRec r{kernel, site, flops, st, g_prof.get(), g_prof.get()};
    (void)hipEventRecord(r.e0, s);
    e1 = r.e1;
    g_prof.recs.push_back(r);
  }
  ~ProfScope() {
    if (e1) (void)hipEventRecord(e1, s);
  }
};
// kern may contain template commas: pass it parenthesised
#define LACT_LAUNCH(kname, site, flops, kern, grid, block, stream, ...)  \
  do {                                                                  \
    ProfScope ps_(kname, site, flops, stream);                          \
    hipLaunchKernelGGL(kern, grid, block, 0, stream, __VA_ARGS__);      \
  } while (0)

#define LACT_LAUNCH_SMEM(kname, site, flops, kern, grid, block, smem_bytes, stream, ...) \
  do {                                                                                   \
    ProfScope ps_(kname, site, flops, stream);                                           \
    hipLaunchKernelGGL(kern, grid, block, smem_bytes, stream, __VA_ARGS__);              \
  } while (0)

// Kernels whose ring exceeds the default dynamic LDS limit opt in once per call site (= instantiation) and device:
// the attribute belongs to the current device.
inline void allow_big_lds(std::atomic<uint64_t>& done, const void* kern, int bytes) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  const uint64_t bit = 1ull << dev;
  if (done.load(std::memory_order_acquire) & bit) return;
  (void)hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  done.fetch_or(bit, std::memory_order_release);
}
#define LACT_BIG_LDS(kern, bytes)                                         \
  do {                                                                    \
    static std::atomic<uint64_t> done_{0};                                \
    allow_big_lds(done_, reinterpret_cast<const void*>(kern), bytes);     \
  } while (0)

template <typename T> const char* tname();
template <> const char* tname<uint16_t>() { return "bf16"; }
template <> const char* tname<float>() { return "f32"; }

#define LACT_CHECK_LAUNCH()                                                     \
  do {                                                                          \
    hipError_t e_ = hipGetLastError();                                          \
    if (e_ != hipSuccess) return fail(std::string("kernel launch failed: ") + hipGetErrorString(e_)); \
  } while (0)

// ---- side stream: the apply steps of a program do not depend on the update chain that runs beside them
// (block-causal: apply(i) and update(i) both read weight version i), so they are enqueued on a second
// stream of default priority, forked from and joined back into the caller's stream with events.  The
// memory-bound tails of one chain then overlap the matrix work of the other.  One stream and one event
// pool per device, created on first use and kept until the process ends.
struct SideCtx {
  hipStream_t stream = nullptr;
  std::vector<hipEvent_t> ev;
  size_t next = 0;
  // Fused Newton-Schulz kernels of this process must not overlap each other (each needs its groups resident as a whole).
  // Launches on one stream follow each other anyway; an event is recorded (on the stream of the newest launch, at the
  // time the next launch arrives) only when that next launch comes from another stream -- a record behind every launch
  // would put ~3 us between the kernel and whatever follows it on the caller's stream.
  hipEvent_t fused_done = nullptr;
  hipStream_t fused_stream = nullptr;
  bool fused_any = false;
  void order_fused_launch(hipStream_t s) {
    if (fused_any && fused_stream != s) {
      if (!fused_done) (void)hipEventCreateWithFlags(&fused_done, hipEventDisableTiming);
      if (hipEventRecord(fused_done, fused_stream) == hipSuccess) {
        (void)hipStreamWaitEvent(s, fused_done, 0);
      } else {   // that stream no longer exists: whatever it still runs is waited for the hard way
        (void)hipGetLastError();
        (void)hipDeviceSynchronize();
      }
    }
    fused_stream = s;
    fused_any = true;
  }
  int cus = 0;                       // compute units of the device (0: not asked yet)
  unsigned* sticky = nullptr;        // device address of this device's count of barrier time-outs
  hipEvent_t event() {
    if (next == ev.size()) {
      hipEvent_t e;
      (void)hipEventCreateWithFlags(&e, hipEventDisableTiming);
      ev.push_back(e);
    }
    return ev[next++];
  }
};
}  // namespace
// Barrier waits of the fused Newton-Schulz kernels that gave up, counted per device since the last
// lact_check_async_error (each GPU holds its own copy; host code reaches it through hipGetSymbolAddress only).
static __device__ unsigned g_async_errors;
namespace {
int g_overlap = 1;          // LACT_OPT_STREAM_OVERLAP: 0 never, 1 where it pays, 2 wherever there is something to overlap
bool g_fused_ns = true;
int g_persist = 1;          // hidden-stage kernels on the persistent engine (LACT_OPT_PERSISTENT_TILES): bit 0 apply, 1 update, 2 apply backward
                            // (the one-tile-per-block kernels of the update and the apply backward, whose pointwise epilogues run on all
                            // eight waves, measured faster than their persistent versions: only the apply's is on by default)
long long g_ns_spin_limit = NS_FUSED_SPIN_LIMIT;   // barrier wait bound of the fused Newton-Schulz kernels (lact_set_option)
std::mutex g_enqueue_mutex;   // one program is enqueued at a time (the side-stream context is shared)
SideCtx* side_ctx() {
  static SideCtx ctx[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  SideCtx& c = ctx[dev];
  if (!c.stream && hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking) != hipSuccess) return nullptr;
  if (c.cus == 0) {
    int n = 0;
    c.cus = (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) ? n : -1;
  }
  if (!c.sticky) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(g_async_errors)) == hipSuccess) c.sticky = static_cast<unsigned*>(ptr);
  }
  c.next = 0;
  return &c;
}

inline char* align256(void* p) { return reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(p) + 255) & ~uintptr_t(255)); }
inline const char* align256(const void* p) {
  return reinterpret_cast<const char*>((reinterpret_cast<uintptr_t>(p) + 255) & ~uintptr_t(255));
}

template <typename T, bool B_KC, int NT, int EPI, bool HALF>
const char* row_gemm_name() {
  static const std::string n = std::string("k_row_gemm<") + tname<T>() + (B_KC ? ",Bkc," : ",Bks,") + std::to_string(NT) +
                               (EPI == EPI_STORE ? ",store" : (EPI == EPI_AXPBY ? ",axpby" : ",axpby_dual")) + (HALF ? ",half>" : ">");
  return n.c_str();
}
template <class TS, int NT, int EPI, bool B_KS>
void launch_row_gemm_dma(const char* site, const RowGemmDmaParams<NT>& q, int batch, hipStream_t s) {
  constexpr int STAGES = row_stages<TS>();
  constexpr int SMEM = cmax(DmaSmem<TS, 1, STAGES>::BYTES, StageTile<TS, 4>::BYTES);
  LACT_BIG_LDS((k_row_gemm_dma<TS, NT, EPI, B_KS>), SMEM);
  static const std::string name = std::string("k_row_gemm_dma<") + std::to_string(TS::BM) + "x" + std::to_string(TS::BN) + "," +
                                  std::to_string(NT) + (EPI == EPI_STORE ? ",store" : (EPI == EPI_AXPBY ? ",axpby" : ",axpby_dual")) +
                                  (B_KS ? ",Bks>" : ",Bkc>");
  RowGemmDmaParams<NT> qq = q;
  qq.map = make_tile_map(ceil_div(q.g.M, TS::BM), ceil_div(q.g.N, TS::BN), batch);
  double ksum = 0;
  for (int t = 0; t < NT; ++t) ksum += q.g.t[t].K;
  LACT_LAUNCH_SMEM(name.c_str(), site, 2.0 * q.g.M * q.g.N * ksum * batch, (k_row_gemm_dma<TS, NT, EPI, B_KS>), dim3(qq.map.grid()),
                   dim3(DMA_THREADS), SMEM, s, qq);
}
int device_cus() {
  static const int cus = [] { int dev = 0, n = 0; (void)hipGetDevice(&dev); return hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256; }();
  return cus;
}
// fp32 launches that would leave a compute unit without a 64 x 64 tile take half tiles instead (gemm_async.h).  us, whole tiles / half: at
// 128 of the former (8 x 512 tokens, d = dh = 128) apply hidden stage 12.1 / 7.4, update 14.8 / 12.2, update backward 24.6 / 18.9, four-term
// row GEMM 17.1 / 13.6; at 192 even; at 384 still 1.1 to 1.15 times faster, but at 256, 512 and 1024 up to 1.4 times slower (two-term row
// GEMM 18.6 / 26.3 at 512), as the half tiles read every A row twice.
bool half_tiles(long long blocks) { return blocks < device_cus(); }
template <typename T, bool B_KC, int NT, int EPI, bool HALF>
void launch_row_gemm_async(const char* site, const RowGemmParams<NT>& p, int batch, hipStream_t s) {
  using AT = AsyncTile<T, HALF>;
  constexpr int SM = AsyncRing<T, 1, HALF>::BYTES;
  const dim3 grid(ceil_div(p.M, AT::TS::BM), ceil_div(p.N, AT::TS::BN), batch);
  double ksum = 0;
  for (int t = 0; t < NT; ++t) ksum += p.t[t].K;
  LACT_BIG_LDS((k_row_gemm<T, B_KC, NT, EPI, HALF>), SM);
  LACT_LAUNCH_SMEM((row_gemm_name<T, B_KC, NT, EPI, HALF>()), site, 2.0 * p.M * p.N * ksum * batch,
                   (k_row_gemm<T, B_KC, NT, EPI, HALF>), grid, dim3(AT::THREADS), SM, s, p);
}
// bf16 with every K a multiple of 16: dedicated-loader kernels; anything else: the small-tile pipeline
template <typename T, bool B_KC, int NT, int EPI>
void launch_row_gemm(const char* site, const RowGemmParams<NT>& p, int batch, hipStream_t s, bool token_rows = false) {
  if constexpr (std::is_same<T, uint16_t>::value) {
    bool ok = p.N % 8 == 0;
    for (int t = 0; t < NT; ++t) ok = ok && p.t[t].K % 16 == 0;
    if (ok) {
      RowGemmDmaParams<NT> q;
      q.g = p;
      q.out_ct = nullptr;
      if (token_rows) {
        // 256 x 128 tiles copy a third fewer operand bytes per FLOP than 128 x 128 ones, but a launch whose blocks fill
        // the last round of compute units only partly wastes more than that: pick by the fuller last round
        const int cus = device_cus();
        auto blocks = [&](int bm, int bn) { return (long long)ceil_div(p.M, bm) * ceil_div(p.N, bn) * batch; };
        auto fill = [&](int bm) { const long long n = blocks(bm, 128); return (double)n / ((double)((n + cus - 1) / cus) * cus); };
        // less than one round: the blocks that fit side by side, down to 128 x 64
        if (blocks(128, 128) <= cus / 2) launch_row_gemm_dma<TS_BWD, NT, EPI, !B_KC>(site, q, batch, s);
        else if (blocks(128, 128) <= cus) launch_row_gemm_dma<TS_SQ, NT, EPI, !B_KC>(site, q, batch, s);
        // (measured at 384 blocks on 256 units: one-term GEMM 27.0 -> 24.5 us with the small tile, two-term GEMM with
        // K-strided weights 34 -> 36 us: only the one-term case switches)
        else if (NT == 1 && fill(256) < 0.8 && fill(128) > fill(256) + 0.1) launch_row_gemm_dma<TS_SQ, NT, EPI, !B_KC>(site, q, batch, s);
        else launch_row_gemm_dma<TS_ROW, NT, EPI, !B_KC>(site, q, batch, s);
      }
      else if (p.M % TS_NS::BM == 0 && p.N % TS_NS::BN == 0) launch_row_gemm_dma<TS_NS, NT, EPI, !B_KC>(site, q, batch, s);
      else launch_row_gemm_dma<TS_SQ, NT, EPI, !B_KC>(site, q, batch, s);
      return;
    }
  }
  if constexpr (!std::is_same<T, uint16_t>::value)
    if (half_tiles((long long)ceil_div(p.M, TSG<T>::BM) * ceil_div(p.N, TSG<T>::BN) * batch)) return launch_row_gemm_async<T, B_KC, NT, EPI, true>(site, p, batch, s);
  launch_row_gemm_async<T, B_KC, NT, EPI, false>(site, p, batch, s);
}

template <int NT>
RowGemmParams<NT> row_params() {
  RowGemmParams<NT> p;
  memset(&p, 0, sizeof(p));
  p.alpha = 1.f;
  return p;
}

inline void set_term(RowGemmTerm& t, const void* A, int lda, long long bsA, const void* B, int ldb, long long bsB, int K) {
  t.A = A; t.lda = lda; t.bsA = bsA; t.B = B; t.ldb = ldb; t.bsB = bsB; t.K = K;
}
inline void set_tr_term(TokenReduceTerm& t, const void* A, int lda, long long bsA, const void* B, int ldb, long long bsB) {
  t.A = A; t.lda = lda; t.bsA = bsA; t.B = B; t.ldb = ldb; t.bsB = bsB;
}

// One Newton-Schulz iteration on n matrices held as [r, c] (always bf16 MFMA, fp32 iterate):
//   A = X X^T;  B = b A + c A A;  X' = a X + B X        (ttt_operation.py:59-62)
struct NsIter {
  int n, r, c, nb_for_mask, mask, plain;
  float ca, cb, cc;
  const float* xf_in; const void* xb_in;           // X: fp32 iterate and its copy in the GEMM type
  void* ab; void* bb;                              // A and B of this iteration (GEMM type)
  void* cab;                                       // c * A (GEMM type): the left operand of (c * A) @ A, a tensor of its own in the reference
  float* xf_out; void* xb_out; float* u_out;       // X': fp32, GEMM type, and fp32 in the original orientation (each nullable)
};
// TN: GEMM operand type of the iteration (bf16 as in the reference, or fp32 for the exact mode)
template <typename TN>
void ns_iteration(const NsIter& I, hipStream_t s) {
  const long long xe = (long long)I.r * I.c, se = (long long)I.r * I.r;
  {
    auto p = row_params<1>();
    set_term(p.t[0], I.xb_in, I.c, xe, I.xb_in, I.c, xe, I.c);
    p.M = I.r; p.N = I.r; p.out = I.ab; p.ldo = I.r; p.bso = se;
    p.out2 = I.cab; p.alpha2 = I.cc;
    launch_row_gemm<TN, true, 1, EPI_STORE>("ns_gram", p, I.n, s);
  }
  {   // B = b * A + (c * A) @ A, ttt_operation.py:60
    auto p = row_params<1>();
    set_term(p.t[0], I.cab, I.r, se, I.ab, I.r, se, I.r);
    p.M = I.r; p.N = I.r; p.out = I.bb; p.ldo = I.r; p.bso = se;
    p.aux = I.ab; p.ldaux = I.r; p.bsaux = se; p.alpha = 1.f; p.beta = I.cb;
    launch_row_gemm<TN, true, 1, EPI_AXPBY>("ns_poly", p, I.n, s);
  }
  {
    auto p = row_params<1>();
    set_term(p.t[0], I.bb, I.r, se, I.xb_in, I.c, xe, I.r);
    p.M = I.r; p.N = I.c; p.ldo = I.c; p.bso = xe;
    p.aux = I.xf_in; p.ldaux = I.c; p.bsaux = xe; p.alpha = 1.f; p.beta = I.ca;
    p.round_out_bf16 = I.plain;
    p.out = I.xf_out; p.out_c = I.xb_out; p.out_t = I.u_out;
    p.transpose_mask = I.mask; p.nb = I.nb_for_mask;
    launch_row_gemm<TN, false, 1, EPI_AXPBY_F32_DUAL>("ns_next", p, I.n, s);
  }
}

template <typename T, typename TN>
struct Runner {
  const Plan& P;
  hipStream_t s;
  char* sv;   // saved
  char* sc;   // scratch
  const lact_desc_t& d;
  hipStream_t s_main, s_side;   // caller's stream; stream of the apply steps (= s_main when overlap is off)
  SideCtx* side = nullptr;
  const size_t* hsel;           // token-major intermediates of the chain being enqueued
  size_t partial_sel;
  Runner(const Plan& p, void* saved, void* scratch, hipStream_t st)
      : P(p), s(st), sv(align256(saved)), sc(align256(scratch)), d(p.d), s_main(st), s_side(st), hsel(p.t_h), partial_sel(p.t_partial) {
    side = side_ctx();
    if (side && !P.groups.empty() && overlap_pays(p, st)) s_side = side->stream;
  }
  // Whether the apply steps on earlier versions run beside the update chain.  What is hidden, against the events of the forks and joins, 60 to
  // 100 us of host time a training step (two forks and a wait for every group) and 6 us on the GPU each, and against the compute units that
  // a group takes from the chain's small launches.  us, overlapped / in line, by 1e9 operations of the apply steps (Plan::side_work), updates
  // and groups:
  //   training, no Newton-Schulz.  2.5, 1, 1 (1024 features) 286 / 345; 2.4, 1, 1 (fp32 384) 252 / 292; 1.0, 5, 1 (512) 487 / 507, but 0.3, 1, 1
  //     (512) 197 / 188 and 0.23, 1, 1 (768) 200 or, on a slower host, 257 / 223: chains of wide matrices are long whatever the tokens.  Up to
  //     256 features 3.5, 1, 1 (192) 238 / 231, 4.0, 4, 2 (96) 395 / 336, 4.4, 5, 2 (128) 417 / 405, but 4.7, 5, 3 (96) 403 / 432, 5.4, 3, 1 (192 x
  //     384) 361 / 384, 7.1, 2, 2 (128) 342 / 385; fp32 5.3, 3, 1 (64) 350 / 311, but 5.6, 2, 1 (96) 321 / 329; and with more groups 3.6, 9, 5 (64) 522 / 538.  Long chains of small links lose at any sum:
  //     2.5, 199, 4 (128) 7683 / 7034; 3.9, 39, 1 (256) 2526 / 2388, but 11.9, 59, 4 (128 x 256) 2976 / 3042.
  //   training with Newton-Schulz.  Matrices of one block (ns_local.h): 2.4, 1, 1 (128) 289 / 278, 2.7, 1, 1 (96) 362 / 336, 4.7, 1, 1 (128)
  //     331 / 363, 5.4, 3, 3 (96) 734 / 745, 4.8, 2, 2 (128 x 256) 584 / 636.  Larger ones of fewer than 128 rows, three launches an iteration:
  //     1.2, 2, 1 (64 x 512) 949 / 852, 4.8, 3, 3 1011 / 996.  The fused kernel of the others leaves units free: 0.27, 1, 1 (192 x 384) 368 / 381,
  //     but 0.2, 1, 1 (256) 319 / 264; long chains 2.9, 29, 1 (256) 6283 / 6187.
  //   forward only.  Half as much to hide, and the host further behind: 7.3, 9, 9 (64) 242 / 214; 11.0, 1, 1 (128 x 256) 112 / 102; 15, 1, 1 (256)
  //     173 / 170, but 10.6, 2, 2 (192) 156 / 167; 33, 9, 3 (384) 485 / 512; 29, 9, 5 (256 x 512) 401 / 408; 2.5, 1, 1 (1024) 100 / 107.  With
  //     Newton-Schulz 5.4, 3, 3 (96) 175 / 171; 2.9, 29, 1 (256) 2761 / 2702; 4.8, 2, 2 (128 x 256) 221 / 224; 7.3, 2, 2 (128 x 384) 284 / 294.
  // A captured call pays no host time.
  static bool overlap_pays(const Plan& P, hipStream_t st) {
    if (g_overlap != 1) return g_overlap > 1;
    const double work = P.side_work, group = work / (double)P.groups.size(), wide = work * P.d.d * P.d.dh;
    const bool many = P.groups.size() >= 4, block_each = P.r <= 128 && P.c <= 256;
    const bool pays = P.d.forward_only ? (P.muon ? work >= 4.5e9 && group >= 2.4e9 : (P.groups.size() >= 2 && group >= 5e9) || wide >= 2.5e15)
                      : work < 1.5e8 * P.nupd ? false
                      : P.muon ? work >= (block_each ? 3e9 : P.r < 128 ? 5e9 : 2.5e8)
                               : work >= (P.bf16 ? 4.6e9 : 5.35e9) || (many && work >= 3e9) || wide >= 2e14;
    if (pays) return true;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cap) == hipSuccess) return cap != hipStreamCaptureStatusNone;
    (void)hipGetLastError();      // (the legacy stream beside another one's capture: the launches will say so)
    return false;
  }
  // ---- fused Newton-Schulz: launches of at most 256 resident blocks
  static bool tiles_fit(int r, int c, int bm, int bn) {
    return r % bm == 0 && r % bn == 0 && c % bn == 0 && r % 64 == 0 && c % 64 == 0 && (r / bm) * (c / bn) <= 32;   // whole K-steps
  }
  // Tile of the fused kernel for a batch: 0 = 192 x 192, 1 = 128 x 128, 2 = 128 x 64, 3 = 128 x 96, -1 = none fits.
  // 192 x 192 when the matrices fill at least half the chip with it, else 128 x 128 (more, smaller blocks), and
  // 128 x 64 or 128 x 96 when even those leave most of the chip idle -- as long as the groups dealt to one XCD (a
  // matrix's blocks share an XCD) still find a compute unit each there.
  static int ns_fused_tile(const NsBatch& B) {
    const bool f192 = tiles_fit(B.r, B.c, 192, 192), f128 = tiles_fit(B.r, B.c, 128, 128), f64 = tiles_fit(B.r, B.c, 128, 64);
    const bool f96 = tiles_fit(B.r, B.c, 128, 96);
    if (f192 && (!f128 || B.n * (B.r / 192) * (B.c / 192) >= 128)) return 0;
    const int per_xcd = (B.n + 7) / 8;
    const bool sparse128 = !f128 || B.n * (B.r / 128) * (B.c / 128) < 128;
    if (f64) {
      const int nbm64 = (B.r / 128) * (B.c / 64);
      if (per_xcd * nbm64 <= 32 && sparse128) return 2;
    }
    if (f96) {
      const int nbm96 = (B.r / 128) * (B.c / 96);
      if (per_xcd * nbm96 <= 32 && sparse128) return 3;
    }
    if (f128) return 1;
    return f192 ? 0 : -1;
  }
  static int ns_fused_nbm(const NsBatch& B) {   // blocks per matrix of the fused kernel
    switch (ns_fused_tile(B)) {
      case 0: return (B.r / 192) * (B.c / 192);
      case 1: return (B.r / 128) * (B.c / 128);
      case 2: return (B.r / 128) * (B.c / 64);
      case 3: return (B.r / 128) * (B.c / 96);
      default: return 0;
    }
  }
  // The fused kernel's groups must be resident as a whole, one block per compute unit, on a device that deals its
  // workgroups to 8 dies of 32 compute units: anything else (a partitioned or smaller device) takes the unfused launches.
  bool ns_fusable(const NsBatch& B) const {
    if (!side || !kNsBf16 || P.S < 1 || P.S > NS_FUSED_MAX_STEPS) return false;
    if (side->cus < 256) return false;
    return ns_fused_tile(B) >= 0;
  }
  bool ns_fused_ok(const NsBatch& B) const { return g_fused_ns && ns_fusable(B); }
  // The unfused launches of a batch the fused kernel could take sum the dot product of the normalisation's backward
  // over the fused kernel's tiles, in its order: switching LACT_OPT_FUSED_NEWTON_SCHULZ then changes no bit.
  bool ns_dot_by_tiles() const { return P.muon && P.nsb.size() == 1 && ns_fusable(P.nsb[0]); }
  template <class TS>
  void launch_ns_dot_tiles_ts(const NsTileDotParams& q, const NsBatch& B) {
    LACT_LAUNCH("k_ns_bwd_dot_tiles", "k_ns_bwd_dot", 0.0, (k_ns_bwd_dot_tiles<TS>), dim3((B.r / TS::BM) * (B.c / TS::BN), B.n), dim3(DMA_THREADS), s, q);
  }
  void launch_ns_dot_tiles(const NsTileDotParams& q, const NsBatch& B) {
    switch (ns_fused_tile(B)) {
      case 0: launch_ns_dot_tiles_ts<TS_NS>(q, B); break;
      case 1: launch_ns_dot_tiles_ts<TS_SQ>(q, B); break;
      case 2: launch_ns_dot_tiles_ts<TS_BWD>(q, B); break;
      case 3: launch_ns_dot_tiles_ts<TS_N96>(q, B); break;
      default: break;
    }
  }
  // Forward only: matrices that fit a compute unit whole (X in LDS: at most 128 x 256) run on one block each.
  bool ns_local_ok(const NsBatch& B) const {
    return g_fused_ns && kNsBf16 && P.S >= 1 && P.S <= NS_FUSED_MAX_STEPS && B.r % 32 == 0 && B.c % 32 == 0 && B.r <= 128 && B.c <= 256;
  }
  template <int RT, int XG>
  void launch_ns_local_t(const NsLocalParams& p, const NsBatch& B) {
    constexpr int SM = ns_local_lds<RT, XG>();
    const double flops = 2.0 * B.r * B.r * (2.0 * B.c + B.r) * P.S * B.n;
    LACT_BIG_LDS((k_ns_local<RT, XG, false>), SM);
    LACT_BIG_LDS((k_ns_local<RT, XG, true>), SM);
    if (d.ns_mode == LACT_NS_PLAIN_BF16) LACT_LAUNCH_SMEM("k_ns_local", "ns_fwd", flops, (k_ns_local<RT, XG, true>), dim3(B.n), dim3(512), SM, s, p);
    else LACT_LAUNCH_SMEM("k_ns_local", "ns_fwd", flops, (k_ns_local<RT, XG, false>), dim3(B.n), dim3(512), SM, s, p);
  }
  void launch_ns_local(NsLocalParams p, const NsBatch& B) {
    p.c = B.c; p.S = P.S; p.nb = B.nb; p.mask = B.mask; p.by_granules = make_udiv(B.c / 8);
    for (int i = 0; i < 3 * P.S; ++i) p.coeffs[i] = P.coeffs[i];
    const bool wide = B.c > 128;
    switch (B.r / 32) {
      case 1: wide ? launch_ns_local_t<1, 32>(p, B) : launch_ns_local_t<1, 16>(p, B); break;
      case 2: wide ? launch_ns_local_t<2, 32>(p, B) : launch_ns_local_t<2, 16>(p, B); break;
      case 3: wide ? launch_ns_local_t<3, 32>(p, B) : launch_ns_local_t<3, 16>(p, B); break;
      default: wide ? launch_ns_local_t<4, 32>(p, B) : launch_ns_local_t<4, 16>(p, B); break;
    }
  }
  // forward: every batch runs in one launch that normalises its matrices itself
  bool ns_fwd_one_launch() const {
    if (!P.muon || P.nsb.empty()) return false;
    for (auto& B : P.nsb)
      if (!ns_local_ok(B) && !ns_fused_ok(B)) return false;
    return true;
  }
  bool ns_fwd_fused_any() const {
    const bool local = ns_fwd_one_launch();   // otherwise the normalisation is a launch of its own and nothing runs local
    for (auto& B : P.nsb)
      if (ns_fused_ok(B) && !(local && ns_local_ok(B))) return true;
    return false;
  }
  // every batch runs fused (and at least one iteration): the Frobenius normalisation's backward is the fused kernel's last stage
  bool ns_all_fused() const {
    if (!P.muon || P.nsb.empty()) return false;
    for (auto& B : P.nsb)
      if (!ns_fused_ok(B)) return false;
    return true;
  }
  bool ns_fused_any() const {
    for (auto& B : P.nsb)
      if (ns_fused_ok(B)) return true;
    return false;
  }
  unsigned* ns_error_word() const { return scr<unsigned>(P.t_nssync) + (size_t)P.g.ns_count() * 32; }
  // barrier lines and error word start at zero: once per Newton-Schulz phase, by the kernel in front of its batches
  ClearWords ns_clear(bool forward) const {
    ClearWords c;
    c.ptr = nullptr; c.n = 0;
    if (P.muon && (forward ? ns_fwd_fused_any() : ns_fused_any())) { c.ptr = scr<unsigned>(P.t_nssync); c.n = P.g.ns_count() * 32 + 32; }
    return c;
  }
  template <class TS, bool BWD>
  void launch_ns_fused_ts(const NsFusedParams& p, const NsBatch& B) {
    using Half = typename NsHalfTile<TS>::type;
    if constexpr (!std::is_void<Half>::value)
      if (B.c >= 2 * B.r) return launch_ns_fused_ts<TS, BWD, Half>(p, B);
    launch_ns_fused_ts<TS, BWD, TS>(p, B);
  }
  template <class TS, bool BWD, class TSQ>
  void launch_ns_fused_ts(NsFusedParams p, const NsBatch& B) {
    constexpr int SM = cmax(cmax(DmaSmem<TS, 1, ns_stages<TS>()>::BYTES, StageTile<TS, 4>::BYTES), DmaSmem<TSQ, 1, ns_stages<TSQ>()>::BYTES);
    LACT_BIG_LDS((k_ns_fused<TS, BWD, TSQ>), SM);
    const int nbm = (B.r / TS::BM) * (B.c / TS::BN);
    const int per = (256 / nbm) / 8 * 8;
    unsigned* sync = scr<unsigned>(P.t_nssync) + (size_t)B.first * 32;
    p.r = B.r; p.c = B.c; p.S = P.S; p.nb = B.nb; p.mask = B.mask;
    for (int i = 0; i < 3 * P.S; ++i) p.coeffs[i] = P.coeffs[i];
    p.error = ns_error_word();
    p.sticky = side->sticky;
    p.spin_limit = g_ns_spin_limit;
    const double terms = BWD ? 6.0 : 3.0;
    auto tile = [](int bm, int bn) { return std::to_string(bm) + "x" + std::to_string(bn); };     // + that of the square stages, where it is another
    static const std::string name = "k_ns_fused<" + tile(TS::BM, TS::BN) + (std::is_same<TS, TSQ>::value ? "" : "+" + tile(TSQ::BM, TSQ::BN)) + (BWD ? ",bwd>" : ",fwd>");
    for (int z0 = 0; z0 < B.n; z0 += per) {
      p.z0 = z0; p.n = std::min(per, B.n - z0); p.sync = sync + (size_t)z0 * 32;
      const int grid = 8 * ((p.n + 7) / 8) * nbm;
      side->order_fused_launch(s);
      LACT_LAUNCH_SMEM(name.c_str(), BWD ? "ns_bwd" : "ns_fwd", terms * 2.0 * B.r * B.r * B.c * P.S * p.n,
                       (k_ns_fused<TS, BWD, TSQ>), dim3(grid), dim3(DMA_THREADS), SM, s, p);
    }
  }
  template <bool BWD>
  void launch_ns_fused(const NsFusedParams& p, const NsBatch& B) {
    switch (ns_fused_tile(B)) {
      case 0: launch_ns_fused_ts<TS_NS, BWD>(p, B); break;
      case 1: launch_ns_fused_ts<TS_SQ, BWD>(p, B); break;
      case 2: launch_ns_fused_ts<TS_BWD, BWD>(p, B); break;
      case 3: launch_ns_fused_ts<TS_N96, BWD>(p, B); break;
      default: break;
    }
  }
  // `waiter` waits for everything enqueued so far on `on`
  void wait_for(hipStream_t waiter, hipStream_t on) {
    if (waiter == on || !side) return;
    hipEvent_t e = side->event();
    (void)hipEventRecord(e, on);
    (void)hipStreamWaitEvent(waiter, e, 0);
  }
  // enqueue on the side chain (its stream and buffers) while this object lives
  struct OnSide {
    Runner& r;
    explicit OnSide(Runner& rr) : r(rr) { r.s = r.s_side; r.hsel = r.P.t_hs; r.partial_sel = r.P.t_partial_side; }
    ~OnSide() { r.s = r.s_main; r.hsel = r.P.t_h; r.partial_sel = r.P.t_partial; }
  };

  float* n0() const { return reinterpret_cast<float*>(sv + P.s_n0); }
  float* wf(int ver) const { return reinterpret_cast<float*>(sv + P.s_wf) + (size_t)ver * P.mat3; }
  T* wc(int ver) const { return reinterpret_cast<T*>(sv + P.s_wc) + (size_t)ver * P.mat3; }
  T* wc(int ver, int j) const { return wc(ver) + (size_t)j * d.b * P.g.elems; }
  // accumulator after `u` updates (pre-norm); main(0) is the initial weight
  float* main_(int u) const { return u == 0 ? wf(0) : reinterpret_cast<float*>(sv + P.s_main) + (size_t)(u - 1) * P.mat3; }
  float* dsave(int u) const { return reinterpret_cast<float*>(sv + P.s_d) + (size_t)u * P.mat3; }
  // momentum state that update `u` starts from: the previous update's, or the one the caller carried in
  bool has_prev(int u) const { return P.momentum && (u > 0 || P.state_in); }
  const float* carried[3] = {nullptr, nullptr, nullptr};    // of a forward call that starts from a state: [b][elems] each
  void mprev(const float* (&m)[3], int u) const {
    if (!has_prev(u)) return;
    for (int j = 0; j < 3; ++j) m[j] = u > 0 ? dsave(u - 1) + (size_t)j * d.b * P.g.elems : carried[j];
  }
  float* mbar(int u) const { return reinterpret_cast<float*>(sv + P.s_mbar) + (size_t)u * d.b; }
  float* usave(int u) const { return reinterpret_cast<float*>(sv + P.s_u) + (size_t)u * P.mat3; }
  TN* g16(int u) const { return reinterpret_cast<TN*>(sv + P.s_g16) + (size_t)u * P.mat3; }
  float* norms(int u) const { return reinterpret_cast<float*>(sv + P.s_norms) + (size_t)u * 3 * d.b; }
  TN* xb(int u, int it) const { return reinterpret_cast<TN*>(sv + P.s_xb) + ((size_t)u * std::max(1, P.S) + it) * P.mat3; }
  size_t sq3() const { return P.sq_total; }
  TN* ab(int u, int it) const { return reinterpret_cast<TN*>(sv + P.s_ab) + ((size_t)u * std::max(1, P.S) + it) * sq3(); }
  TN* bb(int u, int it) const { return reinterpret_cast<TN*>(sv + P.s_bb) + ((size_t)u * std::max(1, P.S) + it) * sq3(); }
  T* h(int i) const { return reinterpret_cast<T*>(sc + hsel[i]); }
  // kept array i (0..2: lr-scaled operands, 3..5: pre-activations) of update u; batch stride pre_bs(u)
  T* pre(int u, int i) const { return reinterpret_cast<T*>(sv + P.s_pre[u]) + (size_t)i * d.b * P.pre_T[u] * d.dh; }
  long long pre_bs(int u) const { return (long long)P.pre_T[u] * d.dh; }
  static constexpr bool kBf16 = std::is_same<T, uint16_t>::value;
  static constexpr bool kNsBf16 = std::is_same<TN, uint16_t>::value;

  // the hidden-stage kernels of the dedicated-loader engine need bf16 and whole 16-element sub-steps
  bool dma_hidden() const { return kBf16 && d.d % 16 == 0; }
  // row-partial slots the update-backward hidden kernel in use writes: (hidden tiles) x (wave columns)
  int lr_parts() const {
    if (!dma_hidden()) return hidden_half(3, P.Tupd, d.b) ? ceil_div(d.dh, 32) : ceil_div(d.dh, TSG<T>::BN) * TSG<T>::WAVES_N;
    if (P.keep_pre) return ceil_div(d.dh, TS_SQ::BN) * TS_SQ::WAVES_N;
    return ceil_div(d.dh, TS_BWD::BN) * TS_BWD::WAVES_N;
  }
  bool hidden_small(int which) const { return which == 0 ? d.d <= 256 : which <= 3 && d.d <= 192; }   // the kernel from kept pre-activations has the large tile only
  // 256 x 128 tiles where their rounds of blocks, one to a compute unit and 1.62 times as long as those of 128 x 128 tiles, take less
  // time (gemm_wide.h).
  bool hidden_wide(int T_, int nz) const {
    if (d.d % 64 || d.d < 384 || d.dh % 8) return false;
    const int cols = ceil_div(d.dh, TS_WIDE::BN) * nz;
    return ceil_div(ceil_div(T_, TS_WIDE::BM) * cols, 256) * 1.62 < ceil_div(ceil_div(T_, 128) * cols, 256);
  }
  // fp32: half tiles (gemm_async.h).  One answer for all updates of a program: it decides where the rates' partial sums lie.
  bool hidden_half(int which, int T_, int nz) const {
    if constexpr (kBf16) return false;
    const int t = which == 3 ? P.Tupd : T_;
    return half_tiles((long long)ceil_div(t, TSG<T>::BM) * ceil_div(d.dh, TSG<T>::BN) * nz);
  }
  // LACT_OPT_PERSISTENT_TILES: its default, the apply alone, gives way to the small tiles; any other mask is taken as it is
  bool hidden_persists(int which) const {
    return d.d % 64 == 0 && ((g_persist >> which) & 1) && side && side->cus > 0 && !(g_persist == 1 && hidden_small(which));
  }
  // steps: steps of the program that the launch covers (apply kernels)
  void launch_hidden(int which, const HiddenParams& hp, int T_, int steps = 1) const {
    const int nz = d.b * steps;
    const double f = (double)T_ * d.d * d.dh * nz;
    if (dma_hidden()) {
      if constexpr (kBf16) {
      HiddenDmaParams q;
      q.h = hp;
      // Tiles.  128 x 128 with three stages, one block per compute unit; where the products are at most three K-steps long
      // (d <= 192) a block's time goes into its first copies and its epilogue, and two smaller blocks per unit overlap
      // theirs.  Measured, us per launch, large / small: 12 heads, d = 128, dh = 256, 4680 tokens: update 52.8 / 46.6,
      // apply backward 46.3 / 42.5, recomputing update backward 96 / 91; d = 96: 27.8 / 25.7, 23.7 / 21.5, 47.9 / 43;
      // d = 256: even; d = 384: update 22.3 / 23.7, apply backward 18.5 / 19.7.  The apply's two accumulators: small tiles up
      // to d = 256 (10.4 / 9.95 at d = 256; persistent blocks on large tiles beyond, where they are alone in running ahead).
      constexpr int SM3 = DmaSmem<TS_SQ, 2, 3>::BYTES;   // the epilogues stage at most three bf16 tiles, inside the ring
      constexpr int SMS = DmaSmem<TS_BWD, 2, 2>::BYTES;
      constexpr int SM6 = cmax(DmaSmem<TS_BWD, 2, 3>::BYTES, 6 * StageTile<TS_BWD, 2>::BYTES);
      constexpr int SM6S = cmax(DmaSmem<TS_64, 2, 3>::BYTES, 6 * StageTile<TS_64, 2>::BYTES);
      LACT_BIG_LDS((k_apply_hidden_dma<TS_SQ>), SM3);
      LACT_BIG_LDS((k_update_hidden_dma<TS_SQ>), SM3);
      LACT_BIG_LDS((k_apply_bwd_hidden_dma<TS_SQ>), SM3);
      LACT_BIG_LDS((k_apply_hidden_dma<TS_BWD, 2, 4>), SMS);
      LACT_BIG_LDS((k_update_hidden_dma<TS_BWD, 2, 4>), SMS);
      LACT_BIG_LDS((k_apply_bwd_hidden_dma<TS_BWD, 2, 4>), SMS);
      LACT_BIG_LDS((k_update_bwd_hidden_dma<TS_BWD>), SM6);
      LACT_BIG_LDS((k_update_bwd_hidden_dma<TS_64, 3, 4>), SM6S);
      LACT_BIG_LDS(k_update_bwd_hidden_kept_dma<TS_SQ>, SM3);
      if (which <= 2 && hidden_persists(which)) {
        HiddenPersistParams hq;
        hq.h = hp; hq.map = make_tile_map(ceil_div(T_, TS_SQ::BM), ceil_div(d.dh, TS_SQ::BN), nz);
        const dim3 gp(persist_grid(hq.map.grid(), side->cus));
        LACT_BIG_LDS(k_hidden_persist<ApplyHiddenPolicy>, PersistLds<ApplyHiddenPolicy>::BYTES);
        LACT_BIG_LDS(k_hidden_persist<UpdateHiddenPolicy>, PersistLds<UpdateHiddenPolicy>::BYTES);
        LACT_BIG_LDS(k_hidden_persist<ApplyBwdHiddenPolicy>, PersistLds<ApplyBwdHiddenPolicy>::BYTES);
        if (which == 0) LACT_LAUNCH_SMEM("k_hidden_persist<apply>", "apply_hidden", 4.0 * f, (k_hidden_persist<ApplyHiddenPolicy>), gp, dim3(DMA_THREADS), PersistLds<ApplyHiddenPolicy>::BYTES, s, hq);
        if (which == 1) LACT_LAUNCH_SMEM("k_hidden_persist<update>", "update_hidden", 6.0 * f, (k_hidden_persist<UpdateHiddenPolicy>), gp, dim3(DMA_THREADS), PersistLds<UpdateHiddenPolicy>::BYTES, s, hq);
        if (which == 2) LACT_LAUNCH_SMEM("k_hidden_persist<apply_bwd>", "apply_bwd_hidden", 6.0 * f, (k_hidden_persist<ApplyBwdHiddenPolicy>), gp, dim3(DMA_THREADS), PersistLds<ApplyBwdHiddenPolicy>::BYTES, s, hq);
        return;
      }
      const bool small = hidden_small(which);
      if ((which == 1 || which == 2) && hidden_wide(T_, nz)) {
        q.map = make_tile_map(ceil_div(T_, TS_WIDE::BM), ceil_div(d.dh, TS_WIDE::BN), nz);
        LACT_BIG_LDS(k_update_hidden_wide, WIDE_LDS);
        LACT_BIG_LDS(k_apply_bwd_hidden_wide, WIDE_LDS);
        const dim3 gw(q.map.grid());
        if (which == 1) LACT_LAUNCH_SMEM("k_update_hidden_wide", "update_hidden", 6.0 * f, k_update_hidden_wide, gw, dim3(DMA_THREADS), WIDE_LDS, s, q);
        else LACT_LAUNCH_SMEM("k_apply_bwd_hidden_wide", "apply_bwd_hidden", 6.0 * f, k_apply_bwd_hidden_wide, gw, dim3(DMA_THREADS), WIDE_LDS, s, q);
        return;
      }
      // tile of the kernel that is launched below: the grid has to cover exactly its tiles
      const int bm = which == 3 && small ? TS_64::BM : 128, bn = which == 3 || small ? 64 : 128;
      static_assert(TS_SQ::BM == 128 && TS_SQ::BN == 128 && TS_BWD::BM == 128 && TS_BWD::BN == 64 && TS_64::BN == 64, "tiles of the hidden-stage kernels");
      q.map = make_tile_map(ceil_div(T_, bm), ceil_div(d.dh, bn), nz);
      const dim3 g(q.map.grid()), t(DMA_THREADS);
      if (which == 0) {
        if (small) LACT_LAUNCH_SMEM("k_apply_hidden_dma", "apply_hidden", 4.0 * f, (k_apply_hidden_dma<TS_BWD, 2, 4>), g, t, SMS, s, q);
        else LACT_LAUNCH_SMEM("k_apply_hidden_dma", "apply_hidden", 4.0 * f, (k_apply_hidden_dma<TS_SQ>), g, t, SM3, s, q);
      } else if (which == 1) {
        if (small) LACT_LAUNCH_SMEM("k_update_hidden_dma", "update_hidden", 6.0 * f, (k_update_hidden_dma<TS_BWD, 2, 4>), g, t, SMS, s, q);
        else LACT_LAUNCH_SMEM("k_update_hidden_dma", "update_hidden", 6.0 * f, (k_update_hidden_dma<TS_SQ>), g, t, SM3, s, q);
      } else if (which == 2) {
        if (small) LACT_LAUNCH_SMEM("k_apply_bwd_hidden_dma", "apply_bwd_hidden", 6.0 * f, (k_apply_bwd_hidden_dma<TS_BWD, 2, 4>), g, t, SMS, s, q);
        else LACT_LAUNCH_SMEM("k_apply_bwd_hidden_dma", "apply_bwd_hidden", 6.0 * f, (k_apply_bwd_hidden_dma<TS_SQ>), g, t, SM3, s, q);
      } else if (which == 3) {
        if (small) LACT_LAUNCH_SMEM("k_update_bwd_hidden_dma", "update_bwd_hidden", 12.0 * f, (k_update_bwd_hidden_dma<TS_64, 3, 4>), g, t, SM6S, s, q);
        else LACT_LAUNCH_SMEM("k_update_bwd_hidden_dma", "update_bwd_hidden", 12.0 * f, (k_update_bwd_hidden_dma<TS_BWD>), g, t, SM6, s, q);
      } else {
        LACT_LAUNCH_SMEM("k_update_bwd_hidden_kept_dma", "update_bwd_hidden", 6.0 * f, (k_update_bwd_hidden_kept_dma<TS_SQ>), g, t, SM3, s, q);
      }
      }
    } else {
      if constexpr (!kBf16)
        if (hidden_half(which, T_, nz)) return launch_hidden_async<true>(which, hp, T_, nz, f);
      launch_hidden_async<false>(which, hp, T_, nz, f);
    }
  }
  template <bool HALF>
  void launch_hidden_async(int which, const HiddenParams& hp, int T_, int nz, double f) const {
    using AT = AsyncTile<T, HALF>;
    constexpr int SM = AsyncRing<T, 2, HALF>::BYTES, SM4 = AsyncRing<T, 4, HALF>::BYTES;
    const dim3 g(ceil_div(T_, AT::TS::BM), ceil_div(d.dh, AT::TS::BN), nz), t(AT::THREADS);
    LACT_BIG_LDS((k_apply_hidden<T, HALF>), SM);
    LACT_BIG_LDS((k_update_hidden<T, HALF>), SM);
    LACT_BIG_LDS((k_apply_bwd_hidden<T, HALF>), SM);
    LACT_BIG_LDS((k_update_bwd_hidden<T, HALF>), SM4);
    if (which == 0) LACT_LAUNCH_SMEM((HALF ? "k_apply_hidden<half>" : "k_apply_hidden"), "apply_hidden", 4.0 * f, (k_apply_hidden<T, HALF>), g, t, SM, s, hp);
    if (which == 1) LACT_LAUNCH_SMEM((HALF ? "k_update_hidden<half>" : "k_update_hidden"), "update_hidden", 6.0 * f, (k_update_hidden<T, HALF>), g, t, SM, s, hp);
    if (which == 2) LACT_LAUNCH_SMEM((HALF ? "k_apply_bwd_hidden<half>" : "k_apply_bwd_hidden"), "apply_bwd_hidden", 6.0 * f, (k_apply_bwd_hidden<T, HALF>), g, t, SM, s, hp);
    if (which == 3) LACT_LAUNCH_SMEM((HALF ? "k_update_bwd_hidden<half>" : "k_update_bwd_hidden"), "update_bwd_hidden", 12.0 * f, (k_update_bwd_hidden<T, HALF>), g, t, SM4, s, hp);
  }
  // An apply step as one kernel, for the head sizes it exists for.  (A value of LACT_OPT_PERSISTENT_TILES other than the default
  // asks for the hidden-stage kernels.)
  template <int D, bool SPLIT>
  void launch_apply_fused(ApplyFusedParams p, int nz) const {
    constexpr int SM = apply_fused_lds<D, SPLIT>();
    LACT_BIG_LDS((k_apply_fused<D, SPLIT>), SM);
    p.map = make_tile_map(ceil_div(p.T, SPLIT ? 128 : 256), 1, nz);
    LACT_LAUNCH_SMEM("k_apply_fused", "apply", 6.0 * p.T * D * p.dh * nz, (k_apply_fused<D, SPLIT>), dim3(p.map.grid()), dim3(512), SM, s, p);
  }
  // Where two waves share 32 tokens (SPLIT, below), the chip is not full and the kernel takes as long as one wave needs for all hidden
  // units, which the kernels in pieces spread over blocks: it loses where there are many of them and few tokens.  us on the GPU (a graph
  // of calls, the initial state's kernel included), in pieces / as one: d = 128, 64 tokens, dh = 128 10.3 / 10.9, 256 10.7 / 14.2, 1024
  // 14.7 / 35.9, 2048 20 / 65; 6 x 1024 tokens, dh = 256 14.6 / 17.0, 512 18.7 / 25.3, 2048 41 / 72; 12 x 1024, dh = 256 18.2 / 19.2; d = 64,
  // 6 x 1024, dh = 512 16.4 / 18.3.  Against that stands one launch less, 3.5 us of host time (calls one after the other, 64 tokens, dh =
  // 64: 14.7 us in pieces, 10.8 as one), which is what a short call is bound by (nvs rendering of 6 x 1024 tokens, dh = 256: 19.5 / 17.7):
  // the one kernel may be that far behind, which it is at 256 hidden units of d = 128.  Whole blocks never lose (dh = 64 to 2048).
  bool apply_fused_pays(int T_, int nz) const {
    const double longer = d.dh / 32 * (0.23 + d.d / 256.0) - 1.05e-6 * T_ * nz * d.dh - 2.2;     // (fitted: 1.3 us off on average)
    return ceil_div(T_, 128) * nz > 256 || longer <= 4;
  }
  bool apply_fused(const HiddenParams& hp, const RowGemmParams<1>& out, int T_, int steps) const {
    if constexpr (kBf16) {
      if (g_persist != 1 || (d.d != 64 && d.d != 96 && d.d != 128) || d.dh % 32 || !apply_fused_pays(T_, d.b * steps)) return false;
      ApplyFusedParams p;
      memset(&p, 0, sizeof(p));
      p.T = T_; p.dh = d.dh;
      p.X = static_cast<const uint16_t*>(hp.X); p.ldx = hp.ldx; p.bsx = hp.bsx; p.gsx = hp.gsx;
      p.W0 = static_cast<const uint16_t*>(hp.W0); p.W1 = static_cast<const uint16_t*>(hp.W1); p.W2 = static_cast<const uint16_t*>(hp.W2);
      p.bsw = hp.bsw; p.gsw = hp.gsw;
      p.out = static_cast<uint16_t*>(out.out); p.ldo = out.ldo; p.bso = out.bso; p.gso = out.gso;
      p.steps = hp.steps;
      const int nz = d.b * steps;
      const bool split = ceil_div(T_, 128) * nz <= 256;
      if (d.d == 64) split ? launch_apply_fused<64, true>(p, nz) : launch_apply_fused<64, false>(p, nz);
      else if (d.d == 96) split ? launch_apply_fused<96, true>(p, nz) : launch_apply_fused<96, false>(p, nz);
      else split ? launch_apply_fused<128, true>(p, nz) : launch_apply_fused<128, false>(p, nz);
      return true;
    }
    return false;
  }
  // Whether the program's updates run as one kernel each (the options that select among the kernels in pieces have their defaults).
  // us per update, in pieces / as one kernel, without Newton-Schulz: 12 heads of 64 with 64 hidden units 128 tokens 16.2 / 11.1, 4096
  // 27.6 / 20.2; 48 heads 128 tokens 20.2 / 14.9, 4096 62.5 / 44.5; 12 heads of 128 with 256 hidden units 128 tokens 22.9 / 18.7, 4096
  // 61.7 / 55.6; 48 heads 42.2 / 40.4 and 281 / 160.  Where Newton-Schulz follows and the matrices are square, the reduction of a short
  // update ends in the momentum step, which the one kernel leaves to a pass of its own (12 heads of 96, 128 tokens 28.5 / 27.1, 512
  // 31.2 / 30.0; 48 heads of 128, 128 tokens 41.0 / 42.3, 512 47.7 / 50.0, 1024 60.3 / 59.8, 4096 157 / 118).
  bool updates_fused() const {
    if (!kBf16 || g_persist != 1 || g_keep_pre >= 0 || P.keep_pre || (d.d != 64 && d.d != 96 && d.d != 128) || d.dh % 32) return false;
    int shortest = INT_MAX, longest = 0;
    for (const auto& st : P.live)
      if (st.kind == LACT_UPDATE) {
        shortest = std::min(shortest, st.end - st.start);
        longest = std::max(longest, st.end - st.start);
      }
    const bool step_in_reduction = P.muon && !P.g.stacked && d.d == d.dh;
    return shortest >= 64 && (!step_in_reduction || longest >= 1024);
  }
  template <int D>
  void launch_update_fused(UpdateFusedParams p, int splits) const {
    constexpr int SM = UpdatePatch<D>::LDS;
    LACT_BIG_LDS((k_update_fused<D>), SM);
    p.map = make_tile_map(splits, p.dh / 32, d.b);
    LACT_LAUNCH_SMEM("k_update_fused", "update", 12.0 * p.T * D * p.dh * d.b, (k_update_fused<D>), dim3(p.map.grid()), dim3(256), SM, s, p);
  }
  // Returns the number of partial-sum slots written.
  int update_fused(const HiddenParams& hp) const {
    if constexpr (kBf16) {
      const Split sp = choose_update_split(hp.T, d.b, d.d, d.dh, P.max_splits(false, 1));
      UpdateFusedParams p;
      memset(&p, 0, sizeof(p));
      p.T = hp.T; p.dh = d.dh; p.split_len = sp.len;
      p.K = static_cast<const uint16_t*>(hp.X); p.ldk = hp.ldx; p.bsk = hp.bsx;
      p.V = static_cast<const uint16_t*>(hp.Y); p.ldv = hp.ldy; p.bsv = hp.bsy;
      p.W0 = static_cast<const uint16_t*>(hp.W0); p.W1 = static_cast<const uint16_t*>(hp.W1); p.W2 = static_cast<const uint16_t*>(hp.W2); p.bsw = hp.bsw;
      p.lr0 = hp.lr0; p.lr1 = hp.lr1; p.lr2 = hp.lr2; p.bslr = hp.bslr;
      p.partial = scr<float>(P.t_partial); p.split_stride = (long long)P.mat3; p.mat_stride = (long long)d.b * P.g.elems;
      if (d.d == 64) launch_update_fused<64>(p, sp.n);
      else if (d.d == 96) launch_update_fused<96>(p, sp.n);
      else launch_update_fused<128>(p, sp.n);
      return sp.n;
    }
    return 0;
  }
  // The hidden stage of an apply's backward and dq as one kernel, for the head sizes it exists for; `dq`: rows of the (first) step.
  template <int D>
  void launch_apply_bwd_fused(ApplyBwdFusedParams p, int nz) const {
    constexpr int SM = ApplyBwdStage<D>::LDS;
    LACT_BIG_LDS((k_apply_bwd_fused<D>), SM);
    p.map = make_tile_map(ceil_div(p.T, 256), 1, nz);
    LACT_LAUNCH_SMEM("k_apply_bwd_fused", "apply_bwd", 10.0 * p.T * D * p.dh * nz, (k_apply_bwd_fused<D>), dim3(p.map.grid()), dim3(512), SM, s, p);
  }
  // us of a training step of four updates and applies with Newton-Schulz, in pieces / as one kernel: 12 x 4096 tokens, 96 x 96 705 / 668,
  // 48 x 1024, 128 x 256 1643 / 1600, 2 x 1024 463 / 477.  A round takes 8 us and 2.4 per 32 hidden units, the hidden stage and dq as kernels of
  // their own 18 us and then by the hidden values (43 + 17 us at 12 x 4680 tokens, d = 128, dh = 256; 35 as one).  With this rule and
  // update_bwd_fused's, steps of four updates and applies of 1 to 48 heads, 64 to 128 features, 64 to 1024 hidden units and 128 to 2048 tokens
  // (219 of them) take at most 1.02 of their time in pieces on the GPU.
  bool apply_bwd_fused(int tokens, int nz) const {
    if (!kBf16 || g_persist != 1 || (d.d != 64 && d.d != 96 && d.d != 128) || d.dh % 32) return false;
    const double pieces = 18 + 45.0 * tokens * nz / (12 * 4680) * d.dh / 256 * (0.5 + d.d / 256.0);
    return 8 + ceil_div(ceil_div(tokens, 256) * nz, 256) * 2.4 * (d.dh / 32) < pieces;
  }
  void apply_bwd_fused(const HiddenParams& hp, T* dq, long long gsd, int nz) const {
    if constexpr (kBf16) {
      auto u16 = [](const void* x) { return static_cast<const uint16_t*>(x); };
      ApplyBwdFusedParams p;
      memset(&p, 0, sizeof(p));
      p.T = hp.T; p.dh = d.dh;
      p.X = u16(hp.X); p.ldx = hp.ldx; p.bsx = hp.bsx; p.gsx = hp.gsx;
      p.Y = u16(hp.Y); p.ldy = hp.ldy; p.bsy = hp.bsy; p.gsy = hp.gsy;
      p.W0 = u16(hp.W0); p.W1 = u16(hp.W1); p.W2 = u16(hp.W2); p.bsw = hp.bsw; p.gsw = hp.gsw;
      p.O0 = static_cast<uint16_t*>(hp.O0); p.O1 = static_cast<uint16_t*>(hp.O1); p.O2 = static_cast<uint16_t*>(hp.O2); p.bso = hp.bso;
      p.dq = reinterpret_cast<uint16_t*>(dq); p.bsd = (long long)d.q_len * d.d; p.gsd = gsd;
      p.steps = hp.steps;
      if (d.d == 64) launch_apply_bwd_fused<64>(p, nz);
      else if (d.d == 96) launch_apply_bwd_fused<96>(p, nz);
      else launch_apply_bwd_fused<128>(p, nz);
    }
  }
  // Whether the backward of the program's updates forms the tokens' gradients in one kernel.  It takes 10 us and, a round of its blocks
  // however few there are, 6 and 3.3 to 4 (d = 64 to 128) per 32 hidden units; the kernels in pieces 17 us and then by the hidden values,
  // more so the longer the products: 126 us at 12 x 4680 tokens, d = 128, dh = 256 (hidden stage 92, token rows beside the reduction 34).
  // us of a training step of four updates and applies (without Newton-Schulz), with this part in pieces / as one kernel: 12 x 4096 tokens,
  // 128 x 256 1195 / 1044, 12 x 256 tokens 337 / 394; 48 x 1024, 64 x 128 630 / 558, 96 x 96 648 / 568.
  bool update_bwd_fused() const {
    if (!kBf16 || g_persist != 1 || g_keep_pre >= 0 || P.keep_pre || (d.d != 64 && d.d != 96 && d.d != 128) || d.dh % 32) return false;
    double pieces = 0, one = 0;
    for (const auto& st : P.live)
      if (st.kind == LACT_UPDATE) {
        const int T_ = st.end - st.start;
        pieces += 17 + 126.0 * d.b * T_ / (12 * 4680) * d.dh / 256 * (0.5 + d.d / 256.0);
        one += 10 + ceil_div(ceil_div(T_, 128) * d.b, 256) * (6 + (2.6 + d.d / 90.0) * (d.dh / 32));
      }
    return one < pieces;
  }
  template <int D>
  void launch_update_bwd_fused(UpdateBwdFusedParams p) const {
    constexpr int SM = BwdStage<D>::LDS;
    LACT_BIG_LDS((k_update_bwd_fused<D>), SM);
    p.map = make_tile_map(ceil_div(p.T, 128), 1, d.b);
    LACT_LAUNCH_SMEM("k_update_bwd_fused", "update_bwd", 24.0 * p.T * D * p.dh * d.b, (k_update_bwd_fused<D>), dim3(p.map.grid()), dim3(256), SM, s, p);
  }
  void update_bwd_fused(const HiddenParams& hp, T* dk, T* dv, long long bsd) const {
    if constexpr (kBf16) {
      auto u16 = [](const void* x) { return static_cast<const uint16_t*>(x); };
      UpdateBwdFusedParams p;
      memset(&p, 0, sizeof(p));
      p.T = hp.T; p.dh = d.dh;
      p.K = u16(hp.X); p.ldk = hp.ldx; p.bsk = hp.bsx;
      p.V = u16(hp.Y); p.ldv = hp.ldy; p.bsv = hp.bsy;
      p.W0 = u16(hp.W0); p.W1 = u16(hp.W1); p.W2 = u16(hp.W2); p.G0 = u16(hp.G0); p.G1 = u16(hp.G1); p.G2 = u16(hp.G2); p.bsw = hp.bsw;
      p.lr0 = hp.lr0; p.lr1 = hp.lr1; p.lr2 = hp.lr2; p.bslr = hp.bslr;
      p.O0 = static_cast<uint16_t*>(hp.O0); p.O1 = static_cast<uint16_t*>(hp.O1); p.O2 = static_cast<uint16_t*>(hp.O2); p.bso = hp.bso;
      p.dk = reinterpret_cast<uint16_t*>(dk); p.dv = reinterpret_cast<uint16_t*>(dv); p.bsd = bsd;
      p.lrpart = hp.lrpart; p.lr_stride = hp.lrpart_mat_stride; p.ldlr = hp.Tupd;
      if (d.d == 64) launch_update_bwd_fused<64>(p);
      else if (d.d == 96) launch_update_bwd_fused<96>(p);
      else launch_update_bwd_fused<128>(p);
    }
  }
  template <typename U> U* scr(size_t off) const { return reinterpret_cast<U*>(sc + off); }

  long long hbs(int T_) const { return (long long)T_ * d.dh; }   // between the batch entries of a step's token-major arrays

  HiddenParams hidden_params(int T_, const void* X, int ldx, long long bsx, const void* Y, int ldy, long long bsy, int ver) const {
    HiddenParams p;
    memset(&p, 0, sizeof(p));
    p.T = T_; p.d = d.d; p.dh = d.dh;
    p.X = X; p.ldx = ldx; p.bsx = bsx;
    p.Y = Y; p.ldy = ldy; p.bsy = bsy;
    p.W0 = wc(ver, 0); p.W1 = wc(ver, 1); p.W2 = wc(ver, 2); p.bsw = P.g.elems;
    p.bso = hbs(T_);
    p.Tupd = P.Tupd;
    return p;
  }

  // The three token-reduction GEMMs of a step.  Returns the number of partial-sum slots written to the scratch
  // buffer (the caller reduces them), or 0 when the result went straight to `add_out` = coeff*add_in + sum.
  // (Either kernel writes straight to add_out when one split covers the tokens.)  bf16, 64 tokens or more: the dedicated-loader
  // kernel (a token count that is not a multiple of 64 ends inside the last K-step, whose surplus rows the loader clears).
  // `prep` (forward update only): d_out / g16 / ss_part / m_prev / mbar of the momentum step; when the whole
  // reduction is one split of the asynchronous-copy kernel, its epilogue does that step and -1 is returned.
  struct PrepFold {
    float* d_out; const float* m_prev[3]; const float* mbar; uint16_t* g16; float* ss_part;
    bool skip_d;
    float* m_ext[3];
    ClearWords clear;
  };
  // `rows`: two token-row GEMMs (four and two terms, dk and dv of an update's backward) that may ride in the same
  // launch as the asynchronous-copy reduction; `done` tells the caller whether they did.
  struct RowCompanions {
    RowGemmParams<4> r4;
    RowGemmParams<2> r2;
    bool done = false;
  };
  template <class TS>
  void launch_tr(const char* site, double flops, dim3 grid, const TokenReduceDmaParams& p) const {
    constexpr int SM = cmax(DmaSmem<TS, 1, row_stages<TS>()>::BYTES, StageTile<TS, 4>::BYTES);
    static const std::string name = "k_token_reduce_dma<" + std::to_string(TS::BM) + "x" + std::to_string(TS::BN) + ">";
    LACT_BIG_LDS(k_token_reduce_dma<TS>, SM);
    LACT_LAUNCH_SMEM(name.c_str(), site, flops, (k_token_reduce_dma<TS>), grid, dim3(DMA_THREADS), SM, s, p);
  }
  template <class TS>
  void launch_tr_rows(const char* site, double flops, dim3 grid, const TokenReduceRowsParams& p) const {
    constexpr int SM = cmax(cmax(DmaSmem<TS_ROW, 1, row_stages<TS_ROW>()>::BYTES, StageTile<TS_ROW, 4>::BYTES),
                            cmax(DmaSmem<TS, 1, row_stages<TS>()>::BYTES, StageTile<TS, 4>::BYTES));
    static const std::string name = "k_token_reduce_rows_dma<" + std::to_string(TS::BM) + "x" + std::to_string(TS::BN) + ">";
    LACT_BIG_LDS(k_token_reduce_rows_dma<TS>, SM);
    LACT_LAUNCH_SMEM(name.c_str(), site, flops, (k_token_reduce_rows_dma<TS>), grid, dim3(DMA_THREADS), SM, s, p);
  }
  int token_reduce(const char* site, const TokenReduceJob (&jobs)[3], int tokens, float* add_out = nullptr,
                   const float* add_in = nullptr, float coeff = 0.f, const PrepFold* prep = nullptr,
                   RowCompanions* rows = nullptr, int steps = 1) const {
    const int mats = 3 * d.b * steps, max_n = P.max_splits(partial_sel == P.t_partial_side, steps);
    TokenReduceParams p;
    memset(&p, 0, sizeof(p));
    for (int i = 0; i < 3; ++i) p.job[i] = jobs[i];
    p.by_nb = make_udiv(d.b); p.mat_elems = P.g.elems;
    float* partial = scr<float>(partial_sel);
    int slots = 0;
    bool direct = false;
    if constexpr (kBf16) {
      if (P.reduce_on_dma(tokens)) {     // a ragged end is handled inside the last K-step
        const int tiles = tr_tiles(d.d, d.dh);
        // with the row GEMMs in the launch the chip is busy: short splits only cost (36.4 us in one split, 38.2 in two, 46.8 in four)
        const Split sp = P.reduce_split(tokens, steps, max_n, rows ? 1536 : P.split_min);
        TokenReduceDmaParams pd;
        static_cast<TokenReduceParams&>(pd) = p;
        pd.tokens = tokens; pd.split_len = sp.len; pd.partial = partial;
        pd.map = make_tile_map(sp.n, tiles, mats);
        for (int j = 0; j < 3; ++j) pd.by_tn[j] = make_udiv(ceil_div(jobs[j].N, tr_big(d.d, d.dh) ? TS_NS::BN : TS_SQ::BN));
        dim3 g(pd.map.grid());
        const double fl = 2.0 * tokens * d.d * d.dh * mats;
        direct = add_out && sp.n == 1;
        const bool folded = prep && sp.n == 1;
        if (folded) {
          pd.prep_d_out = prep->d_out; pd.prep_mbar = prep->mbar; pd.prep_skip_d = prep->skip_d ? 1 : 0;
          pd.prep_g16 = prep->g16; pd.prep_ss_part = prep->ss_part; pd.prep_clear = prep->clear;
          for (int j = 0; j < 3; ++j) { pd.prep_m_prev[j] = prep->m_prev[j]; pd.prep_m_ext[j] = prep->m_ext[j]; }
        } else if (direct) { pd.add_out = add_out; pd.add_in = coeff != 0.f ? add_in : nullptr; pd.coeff = coeff; }
        else slots = sp.n;
        bool with_rows = rows != nullptr && rows->r4.N % 8 == 0 && rows->r2.N % 8 == 0;
        if (with_rows) {
          for (int t = 0; t < 4; ++t) with_rows = with_rows && rows->r4.t[t].K % 16 == 0;
          for (int t = 0; t < 2; ++t) with_rows = with_rows && rows->r2.t[t].K % 16 == 0;
        }
        if (with_rows) {
          TokenReduceRowsParams q;
          q.tr = pd;
          q.r4.g = rows->r4; q.r4.out_ct = nullptr;
          q.r4.map = make_tile_map(ceil_div(rows->r4.M, TS_ROW::BM), ceil_div(rows->r4.N, TS_ROW::BN), d.b);
          q.r2.g = rows->r2; q.r2.out_ct = nullptr;
          q.r2.map = make_tile_map(ceil_div(rows->r2.M, TS_ROW::BM), ceil_div(rows->r2.N, TS_ROW::BN), d.b);
          q.ntr = pd.map.grid(); q.n4 = q.r4.map.grid();
          const dim3 gr(q.ntr + q.n4 + q.r2.map.grid());
          double frows = 0;
          for (int t = 0; t < 4; ++t) frows += 2.0 * rows->r4.M * rows->r4.N * rows->r4.t[t].K * d.b;
          for (int t = 0; t < 2; ++t) frows += 2.0 * rows->r2.M * rows->r2.N * rows->r2.t[t].K * d.b;
          if (tr_big(d.d, d.dh)) launch_tr_rows<TS_NS>(site, fl + frows, gr, q);
          else launch_tr_rows<TS_SQ>(site, fl + frows, gr, q);
          rows->done = true;
        } else if (tr_big(d.d, d.dh)) launch_tr<TS_NS>(site, fl, g, pd);
        else launch_tr<TS_SQ>(site, fl, g, pd);
        return folded ? -1 : slots;
      }
    }
    // fp32, or fewer than 64 tokens
    using TS = TSG<T>;
    constexpr int SM = AsyncRing<T, 1>::BYTES;
    const Split sp = P.reduce_split(tokens, steps, max_n, P.split_min);
    direct = add_out && sp.n == 1;
    if (direct) { p.add_out = add_out; p.add_in = coeff != 0.f ? add_in : nullptr; p.coeff = coeff; }
    p.tokens = tokens; p.split_len = sp.len; p.partial = partial;
    LACT_BIG_LDS(k_token_reduce<T>, SM);
    LACT_LAUNCH_SMEM("k_token_reduce", site, 2.0 * tokens * d.d * d.dh * mats, (k_token_reduce<T>), dim3(P.tiles, sp.n, mats),
                     dim3(TS::THREADS), SM, s, p);
    return direct ? 0 : sp.n;
  }

  Partials partials(size_t buffer, int n) const { return Partials{scr<float>(buffer), n, (long long)P.mat3}; }
  RenormParams renorm_params(int u, int ver_prev) const {
    RenormParams p;
    memset(&p, 0, sizeof(p));
    p.g = P.g;
    const bool replace = P.muon && d.muon_replaces_weight;
    p.base = d.prenorm ? main_(u) : wf(ver_prev);
    p.cw = replace ? 0.f : 1.f;
    p.u = P.muon ? usave(u) : dsave(u);
    p.raw = replace ? dsave(u) : nullptr;
    p.cr = replace ? 1.f : 0.f;
    p.n0 = n0();
    p.weight_norm = d.weight_norm;
    p.u_stacked = (P.muon && P.g.stacked) ? 1 : 0;
    p.eps_in_sqrt = d.renorm_eps_in_sqrt ? 1 : 0;
    return p;
  }

  // ------------------------------------------------------------------------------------------
  int forward(const float* w0, const float* w1, const float* w2, const T* q, const T* k, const T* v, const float* lr0,
              const float* lr1, const float* lr2, const float* mom, T* out, float* const w_out[3], float* const m_out[3],
              const float* const m_in[3]) {
    const dim3 rowgrid(ceil_div(P.g.maxrows(), 4), 3 * d.b);
    // carried momentum state: read where it lies (three copies took 18 us at 3 matrices of 768 x 1536 and two batch entries), but for one
    // that 16-byte loads do not reach (a device-to-device copy node when captured)
    if (P.state_in && P.nupd > 0)
      for (int j = 0; j < 3; ++j) {
        carried[j] = m_in[j];
        if (reinterpret_cast<uintptr_t>(m_in[j]) % 16 == 0) continue;
        char* to = sv + P.s_min + (size_t)j * d.b * P.g.elems * 4;
        if (hipMemcpyAsync(to, m_in[j], (size_t)d.b * P.g.elems * 4, hipMemcpyDeviceToDevice, s) != hipSuccess)
          return fail("copy of the carried momentum state failed");
        carried[j] = reinterpret_cast<const float*>(to);
      }
    {
      InitParams p;
      memset(&p, 0, sizeof(p));
      p.g = P.g; p.w[0] = w0; p.w[1] = w1; p.w[2] = w2; p.nw = P.nw; p.n0 = n0();
      // a call without updates hands the weights back as they are; with bf16 activations nothing else reads the fp32 copy then
      p.wf = (P.bf16 && P.nupd == 0 && d.forward_only) ? nullptr : wf(0);
      p.wc = P.bf16 ? (void*)wc(0) : nullptr;
      if (P.nupd == 0 && w_out)
        for (int j = 0; j < 3; ++j) p.w_ext[j] = w_out[j];
      if (d.w_transposed) LACT_LAUNCH("k_init_state", "k_init_state", 0.0, (k_init_state_transposed<T>), dim3(ceil_div(P.g.maxrows(), 32), 3 * d.b), dim3(256), s, p);
      else LACT_LAUNCH("k_init_state", "k_init_state", 0.0, (k_init_state<T>), rowgrid, dim3(256), s, p);
    }
    // mean of the momentum over the chunk of every update that weighs an earlier state (the first update of a
    // program has none unless the caller carried one in): they depend on the input only -- one launch up front
    if (P.momentum) {
      int u0 = P.state_in ? 0 : 1, ui = 0, n = 0;
      MomentumMeanRanges r;
      auto flush = [&]() {
        if (n > 0) LACT_LAUNCH("k_momentum_mean", "k_momentum_mean", 0.0, k_momentum_mean, dim3(d.b, n), dim3(1024), s, mom, (long long)d.kv_len, r, mbar(u0));
        u0 += n; n = 0;
      };
      for (const auto& st : P.live) {
        if (st.kind != LACT_UPDATE) continue;
        if (ui++ < u0) continue;
        r.start[n] = st.start; r.len[n] = st.end - st.start;
        if (++n == 256) flush();
      }
      flush();
    }
    int ver = 0, u = 0;
    T* upd_z[3] = {nullptr, nullptr, nullptr};   // lr-scaled operands of the current update's gradient GEMMs
    long long upd_zbs = 0;
    bool side_used = false;
    // k * lr0, k * lr2 of all updates in one launch, in line: on a stream of its own, beside the first kernels of the call, the launch
    // itself costs nothing but the two events 7 us on either side and as much host time (us of a training step: eight fp32 heads of
    // 128, 2048 tokens 421 / 411 in line, 6 heads of 256 x 512, 5003 tokens 822 / 809; 16 heads of 384, 4096 tokens 1141 either way; two of 768 x
    // 1536, 60840 tokens 7052 / 7078, which the tokens that updates do not read, left out, more than make up for: 6971).
    const long long klbs = (long long)(P.kl_end - P.kl_begin) * d.d;
    const bool fused = updates_fused();
    if (klbs > 0 && !fused)
      LACT_LAUNCH("k_lr_scale_rows", "update_lr_k", 0.0, (k_lr_scale_rows<T>), dim3((unsigned)(((long long)P.kl_len * d.d / 4 + 255) / 256), d.b, P.kl_ranges), dim3(256), s,
                  k + (size_t)P.kl_begin * d.k_ld, d.k_ld, d.k_bs, lr0 + P.kl_begin, lr2 + P.kl_begin, (long long)d.kv_len, P.kl_end - P.kl_begin, P.kl_period, P.kl_len, d.d,
                  scr<T>(P.t_kl[0]), scr<T>(P.t_kl[1]), klbs);
    // Apply steps only need their weight version.  A group of them is enqueued when its last version is final, on the side stream
    // and at the point of the following update where the chip is least busy -- in front of its Newton-Schulz kernels, which leave
    // a quarter of the compute units idle; the newest version's at the end, on the caller's stream.
    auto apply = [&](const ApplyGroup& g) {
      const int T_ = g.st.end - g.st.start;
      HiddenParams hp = hidden_params(T_, q + (size_t)g.st.start * d.q_ld, d.q_ld, d.q_bs, nullptr, 0, 0, g.ver);
      hp.O0 = h(0);
      auto p = row_params<1>();
      set_term(p.t[0], h(0), d.dh, hbs(T_), wc(g.ver, 1), d.dh, P.g.elems, d.dh);
      p.M = T_; p.N = d.d; p.out = out + (size_t)g.st.out_start * d.o_ld; p.ldo = d.o_ld; p.bso = d.o_bs;
      if (g.n > 1) {
        hp.steps.by_nb = p.steps.by_nb = make_udiv(d.b);
        hp.gsx = (long long)g.dstart * d.q_ld; hp.gsw = (long long)P.mat3;
        p.t[0].gsB = (long long)P.mat3; p.gso = (long long)g.dout * d.o_ld;
      }
      if (apply_fused(hp, p, T_, g.n)) return;
      launch_hidden(0, hp, T_, g.n);
      launch_row_gemm<T, true, 1, EPI_STORE>("apply_out", p, d.b * g.n, s, true);
    };
    size_t next_group = 0;
    auto flush_groups = [&]() {   // those whose versions exist
      size_t end = next_group;
      while (end < P.groups.size() && P.groups[end].ver + P.groups[end].n - 1 <= ver) ++end;
      if (end == next_group) return;
      wait_for(s_side, s_main);
      side_used = true;
      OnSide on_side(*this);
      for (; next_group < end; ++next_group) apply(P.groups[next_group]);
    };
    for (const auto& st : P.live) {
      const int T_ = st.end - st.start;
      if (st.kind == LACT_APPLY) {
        if (ver == P.nupd) apply(ApplyGroup{st, ver, 1, 0, 0});
        continue;
      }
      // ---- update
      const T* kc = k + (size_t)st.start * d.k_ld;
      const T* vc = v + (size_t)st.start * d.v_ld;
      const T* kl0 = scr<T>(P.t_kl[0]) + (size_t)(st.start - P.kl_begin) * d.d;
      const T* kl2 = scr<T>(P.t_kl[1]) + (size_t)(st.start - P.kl_begin) * d.d;
      int dw_slots = 0;
      {
        HiddenParams hp = hidden_params(T_, kc, d.k_ld, d.k_bs, vc, d.v_ld, d.v_bs, ver);
        hp.lr0 = lr0 + st.start; hp.lr1 = lr1 + st.start; hp.lr2 = lr2 + st.start; hp.bslr = d.kv_len;
        // operands of the three gradient GEMMs: dgate_before_act, hidden * lr1, dhidden_before_mul
        T* z0 = h(0); T* z1 = h(1); T* z2 = h(2);
        long long zbs = hbs(T_);
        if (P.keep_pre) {
          // the unscaled operands stay in scratch
          z0 = h(0); z1 = pre(u, 1); z2 = h(2); zbs = pre_bs(u);
          hp.O3 = pre(u, 3); hp.O4 = pre(u, 4); hp.O5 = pre(u, 5);
          hp.O6 = pre(u, 0); hp.O7 = pre(u, 2);
          hp.bso = zbs;
        }
        hp.O0 = z0; hp.O1 = z1; hp.O2 = z2;
        if (fused) dw_slots = update_fused(hp);
        else launch_hidden(1, hp, T_);
        upd_z[0] = z0; upd_z[1] = z1; upd_z[2] = z2; upd_zbs = zbs;
      }
      // the pre-Muon gradient (= the momentum state) of the last update: read by nothing when Newton-Schulz output is
      // what enters the weights (the next update and its backward would read it; the caller gets its own copy)
      const bool d_unread = P.muon && !d.muon_replaces_weight && u + 1 == P.nupd;
      if (!fused) {
        TokenReduceJob jobs[3];
        memset(jobs, 0, sizeof(jobs));
        jobs[0].M = d.dh; jobs[0].N = d.d;
        set_tr_term(jobs[0].t, upd_z[0], d.dh, upd_zbs, kl0, d.d, klbs);
        jobs[1].M = d.d; jobs[1].N = d.dh;
        set_tr_term(jobs[1].t, vc, d.v_ld, d.v_bs, upd_z[1], d.dh, upd_zbs);
        jobs[2].M = d.dh; jobs[2].N = d.d;
        set_tr_term(jobs[2].t, upd_z[2], d.dh, upd_zbs, kl2, d.d, klbs);
        // Muon: the momentum step rides in the reduction's epilogue where one split covers the tokens (every tile exists for every matrix).
        // Three matrices of 768 x 1536 and two batch entries, two of three held transposed: 83 + 24 us as a pass of its own, 98 in it.
        PrepFold pf;
        memset(&pf, 0, sizeof(pf));
        const bool can_fold = kBf16 && kNsBf16 && P.muon && !P.g.stacked;
        if (can_fold) {
          for (int j = 0; j < 3; ++j) pf.m_ext[j] = (u + 1 == P.nupd && P.momentum && m_out) ? m_out[j] : nullptr;
          pf.d_out = dsave(u); mprev(pf.m_prev, u); pf.skip_d = d_unread;
          pf.mbar = has_prev(u) ? mbar(u) : nullptr;
          pf.g16 = reinterpret_cast<uint16_t*>(g16(u)); pf.ss_part = scr<float>(P.t_ss);
          pf.clear.ptr = nullptr; pf.clear.n = 0;
          if (ns_fwd_one_launch()) pf.clear = ns_clear(true);
        }
        dw_slots = token_reduce("update_dw", jobs, T_, nullptr, nullptr, 0.f, can_fold ? &pf : nullptr);
      }
      const bool prep_folded = dw_slots < 0;
      const int ss_parts = prep_folded ? tr_tiles(d.d, d.dh) : P.nblk;
      if (P.muon && !prep_folded) {
        MomentumPrepParams p;
        memset(&p, 0, sizeof(p));
        p.g = P.g; p.dw = partials(P.t_partial, dw_slots);
        mprev(p.m_prev, u);
        p.mbar = has_prev(u) ? mbar(u) : nullptr;
        p.d_out = d_unread ? nullptr : dsave(u);
        p.g16 = g16(u);
        p.ss_part = scr<float>(P.t_ss);
        p.round_partial_bf16 = P.bf16;
        if (u + 1 == P.nupd && P.momentum && m_out)
          for (int j = 0; j < 3; ++j) p.m_ext[j] = m_out[j];
        if (ns_fwd_one_launch()) p.clear = ns_clear(true);
        LACT_LAUNCH("k_momentum_prep", "k_momentum_prep", 0.0, (k_momentum_prep<TN>), dim3(P.nblk, 3 * d.b), dim3(256), s, p);
      }
      flush_groups();
      if (P.muon) {
        const bool scale_in_kernel = ns_fwd_one_launch();
        if (!scale_in_kernel) {
          NsScaleParams p;
          memset(&p, 0, sizeof(p));
          p.g = P.g; p.g16 = g16(u); p.ss_part = scr<float>(P.t_ss); p.nparts = ss_parts; p.norms = norms(u);
          p.xf = scr<float>(P.t_xf[0]); p.xb = xb(u, 0);
          p.u = P.S == 0 ? usave(u) : nullptr;
          p.plain_bf16 = d.ns_mode == LACT_NS_PLAIN_BF16;
          p.clear = ns_clear(true);
          LACT_LAUNCH("k_ns_scale", "k_ns_scale", 0.0, (k_ns_scale<TN>), dim3(P.nblk, P.g.ns_count()), dim3(256), s, p);
        }
        for (const NsBatch& B : P.nsb) {
          if (scale_in_kernel && ns_local_ok(B)) {
            if constexpr (kNsBf16) {
              NsLocalParams f;
              memset(&f, 0, sizeof(f));
              f.g16 = g16(u) + B.xoff;
              f.ss_part = scr<float>(P.t_ss); f.nparts = ss_parts;
              f.part0 = B.first; f.part1 = (P.g.stacked && B.first == 0) ? 2 * d.b : -1;
              f.norms = norms(u) + B.first;
              if (!d.forward_only) {
                f.xb = xb(u, 0) + B.xoff; f.xb_it_stride = (long long)P.mat3;
                f.ab = ab(u, 0) + B.sqoff; f.bb = bb(u, 0) + B.sqoff; f.sq_it_stride = (long long)sq3();
              }
              f.u_out = usave(u) + B.xoff;
              launch_ns_local(f, B);
            }
            continue;
          }
          if (ns_fused_ok(B)) {
            if constexpr (kNsBf16) {
              NsFusedParams f;
              memset(&f, 0, sizeof(f));
              f.plain = d.ns_mode == LACT_NS_PLAIN_BF16;
              f.xf[0] = scr<float>(P.t_xf[0]) + B.xoff; f.xf[1] = scr<float>(P.t_xf[1]) + B.xoff;
              f.xb = xb(u, 0) + B.xoff; f.xb_it_stride = (long long)P.mat3;
              f.ab = ab(u, 0) + B.sqoff; f.bb = bb(u, 0) + B.sqoff; f.sq_it_stride = (long long)sq3();
              f.cab = scr<uint16_t>(P.t_ca) + B.sqoff;
              f.u_out = usave(u) + B.xoff;
              if (scale_in_kernel) {
                f.g16 = reinterpret_cast<const uint16_t*>(g16(u)) + B.xoff;
                f.ss_part = scr<float>(P.t_ss); f.nparts = ss_parts;
                f.part0 = B.first; f.part1 = (P.g.stacked && B.first == 0) ? 2 * d.b : -1;
                f.norms = norms(u) + B.first;
              }
              launch_ns_fused<false>(f, B);
            }
            continue;
          }
          for (int it = 0; it < P.S; ++it) {
            const bool last = it + 1 == P.S;
            NsIter I;
            I.n = B.n; I.r = B.r; I.c = B.c; I.nb_for_mask = B.nb; I.mask = B.mask; I.plain = d.ns_mode == LACT_NS_PLAIN_BF16;
            I.ca = P.coeffs[3 * it]; I.cb = P.coeffs[3 * it + 1]; I.cc = P.coeffs[3 * it + 2];
            I.xf_in = scr<float>(P.t_xf[it & 1]) + B.xoff; I.xb_in = xb(u, it) + B.xoff;
            I.ab = ab(u, it) + B.sqoff; I.bb = bb(u, it) + B.sqoff; I.cab = scr<TN>(P.t_ca) + B.sqoff;
            I.xf_out = last ? nullptr : scr<float>(P.t_xf[(it + 1) & 1]) + B.xoff;
            I.xb_out = last ? (void*)(scr<TN>(P.t_xbtmp) + B.xoff) : (void*)(xb(u, it + 1) + B.xoff);
            I.u_out = last ? usave(u) + B.xoff : nullptr;
            ns_iteration<TN>(I, s);
          }
        }
      }
      {
        RenormParams p = renorm_params(u, ver);
        if (!P.muon) {
          p.dw = partials(P.t_partial, dw_slots);
          p.round_dw_bf16 = P.bf16;
          mprev(p.m_prev, u);
          p.mbar = has_prev(u) ? mbar(u) : nullptr;
          p.d_out = dsave(u);
          if (u + 1 == P.nupd && P.momentum && m_out)
            for (int j = 0; j < 3; ++j) p.m_ext[j] = m_out[j];
        }
        p.main_out = d.prenorm ? main_(u + 1) : nullptr;
        // the fp32 copy of a weight version is the base of the next update (and of its backward): the last one has none
        // (with fp32 activations it is also what the apply steps read)
        p.wf_out = (P.bf16 && u + 1 == P.nupd) ? nullptr : wf(ver + 1);
        p.wc_out = P.bf16 ? (void*)wc(ver + 1) : nullptr;
        if (u + 1 == P.nupd && w_out)
          for (int j = 0; j < 3; ++j) p.w_ext[j] = w_out[j];
        if (P.muon && ns_fwd_fused_any()) p.poison = ns_error_word();
        LACT_LAUNCH("k_update_renorm", "k_update_renorm", 0.0, (k_update_renorm<T>), rowgrid, dim3(256), s, p);
      }
      ++ver;
      ++u;
    }
    if (side_used) wait_for(s_main, s_side);
    // final weights and momentum state: written by the last update's kernels, or by the first kernel when no update runs
    if (m_out && (m_out[0] || m_out[1] || m_out[2])) {
      if (u > 0 && P.momentum) {
      } else
        for (int j = 0; j < 3; ++j)
          if (m_out[j]) LACT_LAUNCH("k_fill_f32", "k_fill_f32", 0.0, k_fill_f32, dim3((unsigned)((d.b * P.g.elems + 255) / 256)), dim3(256), s, m_out[j], 0.f, (long long)d.b * P.g.elems);
    }
    LACT_CHECK_LAUNCH();
    return 0;
  }

  // Threads to a quad of an initial weight's gradient (k_finish_weight_grads): one where every entry has its own, or while the launch has
  // four blocks to a compute unit; else twice as many until it has, up to the entries of a matrix.
  int finish_lanes() const {
    const long long blocks = (P.g.elems / 4 + 255) / 256 * 3 * P.nw;
    int n = 1;
    while (n < 16 && n < d.b / P.nw && blocks * n < 1024) n *= 2;
    return n;
  }

  // ------------------------------------------------------------------------------------------
  // Gradient rows of a token range are stored on first touch and accumulated on a repeat.  `force` (set when two
  // ranges of the program overlap without being equal) pre-zeroes the whole buffer and accumulates everywhere.
  struct Touched {
    std::vector<std::pair<int, int>> seen;
    bool force = false;
    bool accumulate(int a, int b) {
      bool hit = force;
      for (auto& iv : seen) hit = hit || (a < iv.second && iv.first < b);
      seen.emplace_back(a, b);
      return hit;
    }
  };
  // Rows of [0, len) that no step of `kind` touches, and whether any two of its ranges overlap partially.
  static std::vector<std::pair<int, int>> untouched(const std::vector<lact_step_t>& steps, int kind, int len, bool* partial) {
    std::vector<std::pair<int, int>> iv;
    for (auto& st : steps)
      if (st.kind == kind) iv.emplace_back(st.start, st.end);
    *partial = false;
    for (size_t i = 0; i < iv.size(); ++i)
      for (size_t j = i + 1; j < iv.size(); ++j)
        if (iv[i] != iv[j] && iv[i].first < iv[j].second && iv[j].first < iv[i].second) *partial = true;
    std::sort(iv.begin(), iv.end());
    std::vector<std::pair<int, int>> gaps;
    int pos = 0;
    for (auto& r : iv) {
      if (r.first > pos) gaps.emplace_back(pos, r.first);
      pos = std::max(pos, r.second);
    }
    if (pos < len) gaps.emplace_back(pos, len);
    if (*partial) gaps.assign(1, std::make_pair(0, len));
    return gaps;
  }
  struct ZeroList {
    ZeroSegments z;
    int n = 0;
    long long maxlen = 0;
    int nb;
    hipStream_t s;
    bool launched = false;
    ZeroList(int nb_, hipStream_t s_) : nb(nb_), s(s_) {}
    void flush() {
      if (n > 0 && maxlen > 0) {
        LACT_LAUNCH("k_zero_segments", "k_zero_segments", 0.0, k_zero_segments, dim3((unsigned)((maxlen + 4095) / 4096), nb, n), dim3(256), s, z);
        launched = true;
      }
      n = 0; maxlen = 0;
    }
    void add(void* ptr, long long bs, long long off, long long len) {
      if (!ptr || len <= 0) return;
      z.ptr[n] = static_cast<char*>(ptr); z.bs[n] = bs; z.off[n] = off; z.len[n] = len;
      maxlen = std::max(maxlen, len);
      if (++n == 16) flush();
    }
  };

  int backward(const T* q, const T* k, const T* v, const float* lr0, const float* lr1, const float* lr2, const float* mom,
               const T* dout, const float* const dwf[3], float* dw0, float* dw1, float* dw2, T* dq, T* dk, T* dv, float* dlr0,
               float* dlr1, float* dlr2, float* dmom) {
    (void)mom;
    const dim3 rowgrid(ceil_div(P.g.maxrows(), 4), 3 * d.b);
    const dim3 eg((unsigned)((P.g.elems / 4 + 255) / 256), 3 * d.b);
    const dim3 flat((unsigned)((P.mat3 / 4 + 255) / 256));
    float* gwcur = scr<float>(P.t_gwcur);
    float* gn0 = scr<float>(P.t_gn0);
    float* gmcarry = scr<float>(P.t_gmcarry);
    const long long gn0_n = (long long)3 * d.b * P.g.maxrows();
    // gn0 is written (not added to) by the first renorm backward; without any update the final kernel reads zeros
    bool gn0_written = false;
    if (P.nupd == 0) LACT_LAUNCH("k_fill_f32", "k_fill_f32", 0.0, k_fill_f32, dim3((unsigned)((gn0_n + 255) / 256)), dim3(256), s, gn0, 0.f, gn0_n);
    // gradient w.r.t. the current weight version: a full array plus partial sums that its reader (the renorm backward, the final
    // kernel) adds up; nothing of either stands for zero
    struct GradSum {
      const float* base = nullptr; int n = 0;
      bool any() const { return base || n; }
    } gw;
    // another contribution to `g` on the main chain; `rows`: GEMMs that may ride in its launch
    auto contribute = [&](const char* site, const TokenReduceJob (&jobs)[3], int tokens, GradSum& g, RowCompanions* rows) {
      if (g.n) {   // the partial-sum buffer is taken
        LACT_LAUNCH("k_reduce_partials", "k_reduce_partials", 0.0, k_reduce_partials, flat, dim3(256), s, gwcur, g.base, 1.f, scr<float>(P.t_partial), g.n, (long long)P.mat3);
        g = GradSum{gwcur, 0};
      }
      const int n = token_reduce(site, jobs, tokens, gwcur, g.base, g.base ? 1.f : 0.f, nullptr, rows);
      g = n ? GradSum{g.base, n} : GradSum{gwcur, 0};
    };
    if (dwf && (dwf[0] || dwf[1] || dwf[2])) {
      gw.base = gwcur;
      LACT_LAUNCH("k_pack3", "k_pack3", 0.0, k_pack3, eg, dim3(256), s, gwcur, P.g.elems, d.b, dwf[0], dwf[1], dwf[2]);
    }
    // every gradient output is written in full by this call: rows that no step touches are zeroed here.
    // Rows of dq, dk, dv and of the per-token arrays that no step writes are disjoint from everything the steps
    // write: nothing waits for them, and they are cleared on the side stream -- unless ranges overlap partially,
    // where the whole buffers start at zero and every step adds.  The momentum gradient is written by every
    // update but the first of the program (which has no earlier state to weigh).
    Touched seen_q, seen_kv, seen_m;
    const auto gaps_q = untouched(P.live, LACT_APPLY, d.q_len, &seen_q.force);
    const auto gaps_kv = untouched(P.live, LACT_UPDATE, d.kv_len, &seen_kv.force);
    std::vector<lact_step_t> later_updates;
    {
      bool first = true;
      for (auto& st : P.live)
        if (st.kind == LACT_UPDATE) {
          if (!first) later_updates.push_back(st);
          first = false;
        }
    }
    auto gaps_m = untouched(later_updates, LACT_UPDATE, d.kv_len, &seen_m.force);
    if (seen_kv.force) {
      seen_m.force = true;
      gaps_m.assign(1, std::make_pair(0, d.kv_len));
    }
    // momentum gradients: one launch at the end for all updates, unless token ranges of (later) updates repeat
    bool mg_each = seen_m.force;
    for (size_t i = 0; i < later_updates.size() && !mg_each; ++i)
      for (size_t j = i + 1; j < later_updates.size(); ++j)
        if (later_updates[i].start < later_updates[j].end && later_updates[j].start < later_updates[i].end) mg_each = true;
    // learning-rate gradients likewise; every update writes them
    bool lr_each = seen_kv.force;
    {
      std::vector<lact_step_t> ups;
      for (auto& st : P.live)
        if (st.kind == LACT_UPDATE) ups.push_back(st);
      for (size_t i = 0; i < ups.size() && !lr_each; ++i)
        for (size_t j = i + 1; j < ups.size(); ++j)
          if (ups[i].start < ups[j].end && ups[j].start < ups[i].end) lr_each = true;
    }
    std::vector<std::pair<int, int>> lr_ranges;   // met in descending order of the update index, all updates
    const size_t lrslot = (size_t)3 * P.lr_slots * d.b * P.Tupd;
    std::vector<int> mg_updates;
    int mg_parts = P.nblk;   // partial dots per matrix in a momentum-gradient slot (the same for every update)
    std::vector<std::pair<int, int>> mg_ranges;
    // (ranges that repeat add their gradients up)
    const bool bwd_fused = update_bwd_fused() && !lr_each;
    bool q_repeats = seen_q.force;
    for (size_t i = 0; i < P.live.size(); ++i)
      for (size_t j = i + 1; j < P.live.size() && P.live[i].kind == LACT_APPLY; ++j)
        if (P.live[j].kind == LACT_APPLY && P.live[i].start < P.live[j].end && P.live[j].start < P.live[i].end) q_repeats = true;
    auto dq_fused = [&](const ApplyGroup& g) { return !q_repeats && apply_bwd_fused(g.st.end - g.st.start, d.b * g.n); };
    const bool rows_on_side = !seen_q.force && !seen_kv.force && s_side != s_main;
    auto zero_rows = [&](hipStream_t zs) {
      ZeroList zl(d.b, zs);
      const long long rowb = (long long)d.d * sizeof(T);
      for (auto& gp : gaps_q) zl.add(dq, (long long)d.q_len * rowb, gp.first * rowb, (gp.second - gp.first) * rowb);
      for (auto& gp : gaps_kv) {
        zl.add(dk, (long long)d.kv_len * rowb, gp.first * rowb, (gp.second - gp.first) * rowb);
        zl.add(dv, (long long)d.kv_len * rowb, gp.first * rowb, (gp.second - gp.first) * rowb);
        for (float* ptr : {dlr0, dlr1, dlr2})
          zl.add(ptr, (long long)d.kv_len * 4, gp.first * 4LL, (gp.second - gp.first) * 4LL);
      }
      for (auto& gp : gaps_m) zl.add(dmom, (long long)d.kv_len * 4, gp.first * 4LL, (gp.second - gp.first) * 4LL);
      zl.flush();
      return zl.launched;
    };
    if (!rows_on_side) zero_rows(s_main);
    bool side_used = false;
    // Backward of apply steps: weight gradients to full arrays by version (`g.ver` and on; `add`: to what they hold), dq
    auto apply_jobs = [&](const ApplyGroup& g, TokenReduceJob (&jobs)[3]) {
      const int T_ = g.st.end - g.st.start;
      const T* qc = q + (size_t)g.st.start * d.q_ld;
      const T* gc = dout + (size_t)g.st.out_start * d.do_ld;
      memset(jobs, 0, sizeof(jobs));
      jobs[0].M = jobs[2].M = d.dh; jobs[0].N = jobs[2].N = d.d;
      set_tr_term(jobs[0].t, h(1), d.dh, hbs(T_), qc, d.q_ld, d.q_bs);
      jobs[1].M = d.d; jobs[1].N = d.dh;
      set_tr_term(jobs[1].t, gc, d.do_ld, d.do_bs, h(0), d.dh, hbs(T_));
      set_tr_term(jobs[2].t, h(2), d.dh, hbs(T_), qc, d.q_ld, d.q_bs);
      const long long gsh = (long long)d.b * hbs(T_);
      jobs[0].t.gsA = jobs[2].t.gsA = jobs[1].t.gsB = gsh;
      jobs[0].t.gsB = jobs[2].t.gsB = (long long)g.dstart * d.q_ld;
      jobs[1].t.gsA = (long long)g.dout * d.do_ld;
    };
    auto apply_hidden_bwd = [&](const ApplyGroup& g) {
      const int T_ = g.st.end - g.st.start;
      HiddenParams hp = hidden_params(T_, q + (size_t)g.st.start * d.q_ld, d.q_ld, d.q_bs, dout + (size_t)g.st.out_start * d.do_ld, d.do_ld, d.do_bs, g.ver);
      hp.O0 = h(0); hp.O1 = h(1); hp.O2 = h(2);
      if (g.n > 1) {
        hp.steps.by_nb = make_udiv(d.b);
        hp.gsx = (long long)g.dstart * d.q_ld; hp.gsy = (long long)g.dout * d.do_ld; hp.gsw = (long long)P.mat3;
      }
      if (dq_fused(g)) apply_bwd_fused(hp, dq + (size_t)g.st.start * d.d, (long long)g.dstart * d.d, d.b * g.n);
      else launch_hidden(2, hp, T_, g.n);
    };
    auto dq_gemm = [&](const ApplyGroup& g) {   // dq = gY0 W0 + gY2 W2
      if (dq_fused(g)) return;
      const int T_ = g.st.end - g.st.start;
      auto p = row_params<2>();
      set_term(p.t[0], h(1), d.dh, hbs(T_), wc(g.ver, 0), d.d, P.g.elems, d.dh);
      set_term(p.t[1], h(2), d.dh, hbs(T_), wc(g.ver, 2), d.d, P.g.elems, d.dh);
      p.M = T_; p.N = d.d; p.ldo = d.d; p.bso = (long long)d.q_len * d.d;
      int acc = 0;
      std::vector<char> accs(g.n);
      for (int i = 0; i < g.n; ++i) acc += accs[i] = seen_q.accumulate(g.st.start + i * g.dstart, g.st.end + i * g.dstart);
      const bool together = acc == 0 || acc == g.n;
      for (int i = 0; i < (together ? 1 : g.n); ++i) {
        auto pi = p;
        pi.out = dq + (size_t)(g.st.start + i * g.dstart) * d.d;
        pi.accumulate = accs[i];
        if (together && g.n > 1) {
          pi.steps.by_nb = make_udiv(d.b);
          pi.t[0].gsB = pi.t[1].gsB = (long long)P.mat3; pi.gso = (long long)g.dstart * d.d;
        }
        for (int t = 0; t < 2 && i > 0; ++t) {
          pi.t[t].A = (const T*)pi.t[t].A + (size_t)i * d.b * hbs(T_);
          pi.t[t].B = (const T*)pi.t[t].B + (size_t)i * P.mat3;
        }
        launch_row_gemm<T, false, 2, EPI_STORE>("apply_bwd_dq", pi, d.b * (together ? g.n : 1), s, true);
      }
    };
    // The steps on earlier versions need nothing of the chain below: group by group in the order in which the chain asks for them,
    // all enqueued in front of it on the side stream.  `ready[version]`: the newest kernel that its gradient waits for.
    std::vector<float*> gw_side(P.nupd + 1, nullptr);   // null: no apply step on that version
    std::vector<hipEvent_t> ready(P.nupd + 1, nullptr);
    auto apply_groups = [&]() {
      OnSide on_side(*this);
      if (rows_on_side) zero_rows(s);
      for (size_t gi = P.groups.size(); gi-- > 0;) {
        const ApplyGroup& g = P.groups[gi];
        const int T_ = g.st.end - g.st.start;
        side_used = true;
        apply_hidden_bwd(g);
        float* dst = scr<float>(P.t_gwside) + (size_t)P.gw_slot[g.ver] * P.mat3;   // a group's versions have consecutive places
        bool add = false;
        for (int i = 0; i < g.n; ++i) add = add || gw_side[g.ver + i];
        if (add)   // another step on one of these versions came before
          for (int i = 0; i < g.n; ++i)
            if (!gw_side[g.ver + i]) LACT_LAUNCH("k_fill_f32", "k_fill_f32", 0.0, k_fill_f32, dim3((unsigned)((P.mat3 + 255) / 256)), dim3(256), s, dst + i * P.mat3, 0.f, (long long)P.mat3);
        TokenReduceJob jobs[3];
        apply_jobs(g, jobs);
        if (const int n = token_reduce("apply_bwd_dw", jobs, T_, dst, dst, add ? 1.f : 0.f, nullptr, nullptr, g.n)) {
          const long long all = (long long)g.n * P.mat3;
          LACT_LAUNCH("k_reduce_partials", "k_reduce_partials", 0.0, k_reduce_partials, dim3((unsigned)((all / 4 + 255) / 256)), dim3(256), s, dst, add ? dst : nullptr, 1.f, scr<float>(P.t_partial_side), n, all);
        }
        hipEvent_t e = nullptr;
        if (s_side != s_main) {
          e = side->event();
          (void)hipEventRecord(e, s_side);
        }
        for (int i = 0; i < g.n; ++i) { gw_side[g.ver + i] = dst + i * P.mat3; ready[g.ver + i] = e; }
        dq_gemm(g);
      }
    };
    bool groups_started = false;
    hipEvent_t waited = nullptr;
    int ver = P.nupd, u = P.nupd;
    int carry_main = -1;       // index of the gwhat buffer holding the accumulator's gradient (pre-norm)
    bool gm_valid = false;     // gmcarry holds d loss / d (momentum state after update u-1)
    for (int si = (int)P.live.size() - 1; si >= 0; --si) {
      const lact_step_t& st = P.live[si];
      const int T_ = st.end - st.start;
      if (st.kind == LACT_APPLY) {
        if (ver < P.nupd) continue;   // in a group
        // Applies of the newest weight version: the update chain cannot start before their weight gradients, so they stay on the
        // caller's stream; only the last one's dq, which nothing waits for, goes to the side stream (its operands have buffers of
        // their own).
        const ApplyGroup g{st, ver, 1, 0, 0};
        hsel = P.t_hn;
        apply_hidden_bwd(g);
        TokenReduceJob jobs[3];
        apply_jobs(g, jobs);
        contribute("apply_bwd_dw", jobs, T_, gw, nullptr);
        const bool last = si == 0 || P.live[si - 1].kind == LACT_UPDATE;
        if (last && s_side != s_main) {
          wait_for(s_side, s_main);
          groups_started = side_used = true;
          s = s_side;
        }
        dq_gemm(g);
        s = s_main;
        hsel = P.t_h;
        if (groups_started) apply_groups();
        continue;
      }
      if (!groups_started) {
        groups_started = true;
        wait_for(s_side, s_main);
        apply_groups();
      }
      // ---- update u-1: weights ver-1 -> ver
      --u;
      const int vprev = ver - 1;
      const int gw_idx = carry_main == 0 ? 1 : 0;
      float* gwhat = scr<float>(P.t_gwhat[gw_idx]);
      const bool carry_here = P.momentum && (u > 0 || gm_valid);
      const size_t mslot = (size_t)3 * d.b * P.mdot_parts;   // partial momentum dots of one update
      int cur = 0;  // which gxf/gxb buffer holds the running Newton-Schulz gradient
      {
        RenormParams p = renorm_params(u, vprev);
        p.gy = gw.base;
        p.gyp = partials(P.t_partial, gw.n);
        if (ready[ver] && ready[ver] != waited) {   // for the weight gradients only: dq GEMMs may still be running
          waited = ready[ver];
          (void)hipStreamWaitEvent(s_main, waited, 0);
        }
        p.gy2 = gw_side[ver];
        p.carry_in = (d.prenorm && carry_main >= 0) ? scr<float>(P.t_gwhat[carry_main]) : nullptr;
        p.gw_hat = gwhat;
        p.gn0 = gn0; p.gn0_init = !gn0_written;
        gn0_written = true;
        p.clear = ns_clear(false);
        const bool as_they_lie = P.g.x_contiguous(0) && P.g.x_contiguous(1) && P.g.x_contiguous(2);
        if (P.muon) {
          if (as_they_lie) { p.gxf = scr<float>(P.t_gxf[0]); p.gxb = scr<TN>(P.t_gxb[0]); }
        } else {
          p.gc = scr<T>(P.t_gc);
          p.gm_carry = carry_here ? gmcarry : nullptr; p.carry_valid = gm_valid; p.carry_write = u > 0;
          if (P.momentum && u > 0) {
            mprev(p.m_prev, u); p.mbar = mbar(u);
            p.mdot_part = scr<float>(P.t_mdot) + (size_t)u * mslot;
          }
        }
        LACT_LAUNCH("k_renorm_bwd", "k_renorm_bwd", 0.0, (k_renorm_bwd<T, TN>), rowgrid, dim3(256), s, p);
        if (P.muon && !as_they_lie)   // whole segments through LDS instead of two and four bytes at a time
          LACT_LAUNCH("k_to_ns_orientation", "k_to_ns_orientation", 0.0, (k_to_ns_orientation<TN>), dim3(P.nblk, 3 * d.b), dim3(256), s, P.g, gwhat, scr<float>(P.t_gxf[0]), (void*)scr<TN>(P.t_gxb[0]));
      }
      if (d.prenorm) carry_main = gw_idx;
      // The backward of the Frobenius normalisation as the fused kernel's last stages: the partial dots always
      // (one batch, every matrix fused); the gradient in the compute type too when nothing else enters it (no
      // momentum state to carry, no raw-gradient term) and every matrix is held as it lies (square shapes).
      const bool dot_in_kernel = ns_all_fused() && P.nsb.size() == 1;
      const bool prep_in_kernel = dot_in_kernel && kBf16 && !(P.muon && d.muon_replaces_weight) &&
                                  P.g.x_contiguous(0) && P.g.x_contiguous(1) && P.g.x_contiguous(2);
      if (P.muon) {
        for (const NsBatch& B : P.nsb) {
          const int n = B.n, r = B.r, c = B.c;
          const long long xe = (long long)r * c, se = (long long)r * r;
          TN* sg = scr<TN>(P.t_sg) + B.sqoff;
          TN* gas = scr<TN>(P.t_gas) + B.sqoff;
          if (ns_fused_ok(B)) {
            if constexpr (kNsBf16) {
              NsFusedParams f;
              memset(&f, 0, sizeof(f));
              f.xb = xb(u, 0) + B.xoff; f.xb_it_stride = (long long)P.mat3;
              f.ab = ab(u, 0) + B.sqoff; f.bb = bb(u, 0) + B.sqoff; f.sq_it_stride = (long long)sq3();
              f.gxf[0] = scr<float>(P.t_gxf[0]) + B.xoff; f.gxf[1] = scr<float>(P.t_gxf[1]) + B.xoff;
              f.gxb[0] = scr<uint16_t>(P.t_gxb[0]) + B.xoff; f.gxb[1] = scr<uint16_t>(P.t_gxb[1]) + B.xoff;
              f.sg = reinterpret_cast<uint16_t*>(sg); f.gas = reinterpret_cast<uint16_t*>(gas);
              if (dot_in_kernel) {
                f.g16 = reinterpret_cast<const uint16_t*>(g16(u)) + B.xoff;
                f.dot_part = scr<float>(P.t_dot);
                f.norms = norms(u) + B.first;
                if (prep_in_kernel) {
                  f.gc = scr<uint16_t>(P.t_gc) + B.xoff;
                  if (carry_here) {   // as in k_grad_prep
                    f.gm_carry = gmcarry; f.carry_valid = gm_valid; f.carry_write = u > 0;
                    f.m_prev = u > 0 ? dsave(u - 1) : nullptr;
                    f.mbar = u > 0 ? mbar(u) : nullptr;
                    f.mdot_part = scr<float>(P.t_mdot) + (size_t)u * mslot;
                  }
                }
              }
              launch_ns_fused<true>(f, B);
            }
            continue;
          }
          int bc = 0;   // every batch starts from buffer 0 and ends in buffer S & 1
          for (int it = P.S - 1; it >= 0; --it) {
            const float ca = P.coeffs[3 * it], cb = P.coeffs[3 * it + 1], cc = P.coeffs[3 * it + 2];
            TN* gb = scr<TN>(P.t_gxb[bc]) + B.xoff;
            float* gf = scr<float>(P.t_gxf[bc]) + B.xoff;
            TN* xk = xb(u, it) + B.xoff;
            TN* ak = ab(u, it) + B.sqoff;
            TN* bk = bb(u, it) + B.sqoff;
            {  // Sg = G X^T + X G^T
              auto p = row_params<2>();
              set_term(p.t[0], gb, c, xe, xk, c, xe, c);
              set_term(p.t[1], xk, c, xe, gb, c, xe, c);
              p.M = r; p.N = r; p.out = sg; p.ldo = r; p.bso = se;
              launch_row_gemm<TN, true, 2, EPI_STORE>("ns_bwd_sg", p, n, s);
            }
            {  // gA + gA^T = b Sg + c (Sg A + A Sg)
              auto p = row_params<2>();
              set_term(p.t[0], sg, r, se, ak, r, se, r);
              set_term(p.t[1], ak, r, se, sg, r, se, r);
              p.M = r; p.N = r; p.out = gas; p.ldo = r; p.bso = se;
              p.aux = sg; p.ldaux = r; p.bsaux = se; p.alpha = cc; p.beta = cb;
              launch_row_gemm<TN, true, 2, EPI_AXPBY>("ns_bwd_ga", p, n, s);
            }
            {  // gX = a G + B G + (gA + gA^T) X
              auto p = row_params<2>();
              set_term(p.t[0], bk, r, se, gb, c, xe, r);
              set_term(p.t[1], gas, r, se, xk, c, xe, r);
              p.M = r; p.N = c; p.ldo = c; p.bso = xe;
              p.aux = gf; p.ldaux = c; p.bsaux = xe; p.alpha = 1.f; p.beta = ca;
              p.out = scr<float>(P.t_gxf[bc ^ 1]) + B.xoff;
              p.out_c = scr<TN>(P.t_gxb[bc ^ 1]) + B.xoff;
              launch_row_gemm<TN, false, 2, EPI_AXPBY_F32_DUAL>("ns_bwd_gx", p, n, s);
            }
            bc ^= 1;
          }
        }
        cur = P.S & 1;
        if (!dot_in_kernel && ns_dot_by_tiles()) {
          if constexpr (kNsBf16) {
            const NsBatch& B = P.nsb[0];
            NsTileDotParams q;
            q.gx = scr<float>(P.t_gxf[cur]) + B.xoff; q.g16 = reinterpret_cast<const uint16_t*>(g16(u)) + B.xoff;
            q.dot_part = scr<float>(P.t_dot); q.r = B.r; q.c = B.c;
            launch_ns_dot_tiles(q, B);
          }
        } else if (!dot_in_kernel) {
          NsDotParams dp;
          dp.g = P.g; dp.gx0 = scr<float>(P.t_gxf[cur]); dp.g16 = g16(u); dp.dot_part = scr<float>(P.t_dot);
          LACT_LAUNCH("k_ns_bwd_dot", "k_ns_bwd_dot", 0.0, (k_ns_bwd_dot<TN>), dim3(P.nblk, P.g.ns_count()), dim3(256), s, dp);
        }
      }
      if (P.muon && !prep_in_kernel) {
        GradPrepParams p;
        memset(&p, 0, sizeof(p));
        p.g = P.g;
        p.gx0 = scr<float>(P.t_gxf[cur]); p.g16 = g16(u); p.norms = norms(u);
        p.dot_part = scr<float>(P.t_dot); p.nparts = (dot_in_kernel || ns_dot_by_tiles()) ? ns_fused_nbm(P.nsb[0]) : P.nblk;
        p.gw_hat = gwhat; p.cr = d.muon_replaces_weight ? 1.f : 0.f;
        p.gm_carry = carry_here ? gmcarry : nullptr; p.carry_valid = gm_valid;
        p.carry_write = u > 0;
        p.m_prev = (P.momentum && u > 0) ? dsave(u - 1) : nullptr;
        p.mbar = (P.momentum && u > 0) ? mbar(u) : nullptr;
        p.gc = scr<T>(P.t_gc);
        p.mdot_part = scr<float>(P.t_mdot) + (size_t)u * mslot;
        if (ns_fused_any()) p.poison = ns_error_word();
        LACT_LAUNCH("k_grad_prep", "k_grad_prep", 0.0, (k_grad_prep<T, TN>), dim3(P.nblk, 3 * d.b), dim3(256), s, p);
      }
      if (P.momentum) {
        gm_valid = true;
        // partial momentum dots per matrix: one per block of the kernel that formed them, or one per tile of the fused kernel
        mg_parts = !P.muon ? (int)rowgrid.x : prep_in_kernel ? ns_fused_nbm(P.nsb[0]) : P.nblk;
        // the gradient of the per-token momentum needs these dot products only: written by one launch at the end
        // (by one launch per update, in this order, when token ranges repeat and their shares add up)
        if (u > 0) {
          const bool acc = seen_m.accumulate(st.start, st.end);
          if (acc || mg_each) {
            MomentumMeanRanges r1;
            r1.start[0] = st.start; r1.len[0] = T_;
            LACT_LAUNCH("k_momentum_grad", "k_momentum_grad", 0.0, k_momentum_grad, dim3(d.b, 1), dim3(256), s, scr<float>(P.t_mdot) + (size_t)u * mslot,
                        0LL, mg_parts, d.b, dmom, (long long)d.kv_len, r1, acc ? 1 : 0);
          } else {
            mg_updates.push_back(u);
            mg_ranges.emplace_back(st.start, T_);
          }
        }
      }
      const T* kc = k + (size_t)st.start * d.k_ld;
      const T* vc = v + (size_t)st.start * d.v_ld;
      T* gcm = scr<T>(P.t_gc);
      T* g0 = gcm; T* g1 = gcm + (size_t)d.b * P.g.elems; T* g2 = gcm + (size_t)2 * d.b * P.g.elems;
      // lr-scaled operands of the forward's gradient GEMMs: kept by the forward, or written again by the hidden kernel
      T* z0 = h(3); T* z1 = h(4); T* z2 = h(5);
      long long zbs = hbs(T_);
      {
        HiddenParams hp = hidden_params(T_, kc, d.k_ld, d.k_bs, vc, d.v_ld, d.v_bs, vprev);
        hp.lr0 = lr0 + st.start; hp.lr1 = lr1 + st.start; hp.lr2 = lr2 + st.start; hp.bslr = d.kv_len;
        hp.G0 = g0; hp.G1 = g1; hp.G2 = g2;
        hp.O0 = h(0); hp.O1 = h(1); hp.O2 = h(2); hp.O3 = h(3); hp.O4 = h(4); hp.O5 = h(5);
        hp.lrpart = scr<float>(P.t_lrpart) + (size_t)u * lrslot;
        hp.lrpart_stride = (long long)d.b * P.Tupd;
        hp.lrpart_mat_stride = (long long)P.lr_slots * d.b * P.Tupd;
        if (P.keep_pre) {
          hp.I0 = pre(u, 3); hp.I1 = pre(u, 4); hp.I2 = pre(u, 5); hp.bsi = pre_bs(u);
          hp.O3 = hp.O4 = hp.O5 = nullptr;
          z0 = pre(u, 0); z1 = pre(u, 1); z2 = pre(u, 2); zbs = pre_bs(u);
        }
        if (bwd_fused) update_bwd_fused(hp, dk + (size_t)st.start * d.d, dv + (size_t)st.start * d.d, (long long)d.kv_len * d.d);
        else launch_hidden(P.keep_pre ? 4 : 3, hp, T_);
      }
      const bool acc_kv = seen_kv.accumulate(st.start, st.end);
      // dk and dv share the launch of the token reduction below (when it runs on the asynchronous-copy kernel; otherwise they are
      // launched after it).  Measured against a stream of their own beside the rest of the chain: 2.32 against 2.45 ms with 216
      // reduction blocks per update, 2.87 against 3.12 ms with 48; the hand-over costs more than what they fill.
      RowCompanions rows_job;
      {  // dk = (dgate*lr0) G0 + (dh2*lr2) G2 + gG W0 + gH2 W2
        auto p = row_params<4>();
        set_term(p.t[0], z0, d.dh, zbs, g0, d.d, P.g.elems, d.dh);
        set_term(p.t[1], z2, d.dh, zbs, g2, d.d, P.g.elems, d.dh);
        set_term(p.t[2], h(0), d.dh, hbs(T_), wc(vprev, 0), d.d, P.g.elems, d.dh);
        set_term(p.t[3], h(2), d.dh, hbs(T_), wc(vprev, 2), d.d, P.g.elems, d.dh);
        p.M = T_; p.N = d.d; p.out = dk + (size_t)st.start * d.d; p.ldo = d.d; p.bso = (long long)d.kv_len * d.d;
        p.accumulate = acc_kv;
        rows_job.r4 = p;
      }
      {  // dv = (hidden*lr1) G1^T + gDH W1^T
        auto p = row_params<2>();
        set_term(p.t[0], z1, d.dh, zbs, g1, d.dh, P.g.elems, d.dh);
        set_term(p.t[1], h(1), d.dh, hbs(T_), wc(vprev, 1), d.dh, P.g.elems, d.dh);
        p.M = T_; p.N = d.d; p.out = dv + (size_t)st.start * d.d; p.ldo = d.d; p.bso = (long long)d.kv_len * d.d;
        p.accumulate = acc_kv;
        rows_job.r2 = p;
      }
      // learning-rate gradients: row partials of every update kept, one reduction launch at the end (one launch per
      // update, in this order, when token ranges repeat and their shares add up)
      if (lr_each) {
        MomentumMeanRanges r1;
        r1.start[0] = st.start; r1.len[0] = T_;
        LACT_LAUNCH("k_lr_reduce", "k_lr_reduce", 0.0, k_lr_reduce, dim3(ceil_div(T_, 256), d.b, 3), dim3(256), s,
                    scr<float>(P.t_lrpart) + (size_t)u * lrslot, 0LL, (long long)P.lr_slots * d.b * P.Tupd, (long long)d.b * P.Tupd, bwd_fused ? 1 : lr_parts(),
                    P.Tupd, dlr0, dlr1, dlr2, (long long)d.kv_len, r1, acc_kv ? 1 : 0);
      } else {
        lr_ranges.emplace_back(st.start, T_);
      }
      {
        TokenReduceJob jobs[3];
        memset(jobs, 0, sizeof(jobs));
        jobs[0].M = d.dh; jobs[0].N = d.d;
        set_tr_term(jobs[0].t, h(0), d.dh, hbs(T_), kc, d.k_ld, d.k_bs);
        jobs[1].M = d.d; jobs[1].N = d.dh;
        set_tr_term(jobs[1].t, vc, d.v_ld, d.v_bs, h(1), d.dh, hbs(T_));
        jobs[2].M = d.dh; jobs[2].N = d.d;
        set_tr_term(jobs[2].t, h(2), d.dh, hbs(T_), kc, d.k_ld, d.k_bs);
        // the update before: its weights enter these as they are, unless Newton-Schulz output replaces them or an accumulator carries on
        gw = GradSum{(d.prenorm || (P.muon && d.muon_replaces_weight)) ? nullptr : gwhat, 0};
        contribute(kBf16 && !bwd_fused ? "update_bwd_dw_dk_dv" : "update_bwd_dw", jobs, T_, gw, bwd_fused ? nullptr : &rows_job);
        if (!bwd_fused && !rows_job.done) {
          launch_row_gemm<T, false, 4, EPI_STORE>("update_bwd_dk", rows_job.r4, d.b, s, true);
          launch_row_gemm<T, true, 2, EPI_STORE>("update_bwd_dv", rows_job.r2, d.b, s, true);
        }
      }
      --ver;
    }
    if (!lr_ranges.empty()) {
      const int total = (int)lr_ranges.size();   // = updates; entry total - 1 - u belongs to update u
      for (int u0 = 0; u0 < total; u0 += 256) {
        const int n = std::min(256, total - u0);
        MomentumMeanRanges r;
        int longest = 0;
        for (int i = 0; i < n; ++i) {
          r.start[i] = lr_ranges[total - 1 - (u0 + i)].first; r.len[i] = lr_ranges[total - 1 - (u0 + i)].second;
          longest = std::max(longest, r.len[i]);
        }
        LACT_LAUNCH("k_lr_reduce", "k_lr_reduce", 0.0, k_lr_reduce, dim3(ceil_div(longest, 256), d.b, 3 * n), dim3(256), s,
                    scr<float>(P.t_lrpart) + (size_t)u0 * lrslot, (long long)lrslot, (long long)P.lr_slots * d.b * P.Tupd, (long long)d.b * P.Tupd,
                    bwd_fused ? 1 : lr_parts(), P.Tupd, dlr0, dlr1, dlr2, (long long)d.kv_len, r, 0);
      }
    }
    if (!mg_updates.empty()) {
      // deferred updates are all updates but the first, met in descending order: slot u - 1 of the launch is update u
      const size_t slot = (size_t)3 * d.b * P.mdot_parts;
      const int total = (int)mg_updates.size();
      for (int i0 = 0; i0 < total; i0 += 256) {
        const int n = std::min(256, total - i0);
        MomentumMeanRanges r;
        int umin = mg_updates[total - 1 - i0];
        for (int i = 0; i < n; ++i) {
          const int idx = total - 1 - (i0 + i);   // ascending update index
          r.start[i] = mg_ranges[idx].first; r.len[i] = mg_ranges[idx].second;
        }
        LACT_LAUNCH("k_momentum_grad", "k_momentum_grad", 0.0, k_momentum_grad, dim3(d.b, n), dim3(256), s, scr<float>(P.t_mdot) + (size_t)umin * slot,
                    (long long)slot, mg_parts, d.b, dmom, (long long)d.kv_len, r, 0);
      }
    }
    {
      FinishParams p;
      memset(&p, 0, sizeof(p));
      if (side_used) wait_for(s_main, s_side);
      p.g = P.g; p.gw = gw.base; p.gwp = partials(P.t_partial, gw.n);
      p.gw2 = gw_side[0];
      p.carry = (d.prenorm && carry_main >= 0) ? scr<float>(P.t_gwhat[carry_main]) : nullptr;
      p.gn0 = gn0; p.n0 = n0(); p.w_init = wf(0);
      p.through_norms = d.detach_norms ? 0 : 1;
      p.out[0] = dw0; p.out[1] = dw1; p.out[2] = dw2; p.nw = P.nw; p.lanes = finish_lanes();
      LACT_LAUNCH("k_finish_weight_grads", "k_finish_weight_grads", 0.0, k_finish_weight_grads, dim3((unsigned)((P.g.elems / 4 * p.lanes + 255) / 256), 3 * P.nw), dim3(256), s, p);
    }
    LACT_CHECK_LAUNCH();
    return 0;
  }
};

int check_ptrs(std::initializer_list<const void*> ps, const char* what) {
  for (const void* p : ps)
    if (!p) return fail(std::string("null pointer: ") + what);
  return 0;
}

}  // namespace

// ---- standalone Newton-Schulz ---------------------------------------------------------------
namespace {
struct NsPlan {
  MatGeom g;
  int r, c, nblk;
  size_t o_g16, o_ss, o_norm, o_xf[2], o_xb[2], o_ab, o_bb, o_ca, bytes;
  void build(int n, int rows, int cols) {
    // one "matrix kind" (index 0) of shape [rows, cols]: d = cols, dh = rows
    g.d = cols; g.dh = rows; g.nb = n; g.elems = (long long)rows * cols; g.stacked = 0;
    r = std::min(rows, cols); c = std::max(rows, cols);
    nblk = std::max(1, std::min(256, (int)((g.elems + 2047) / 2048)));
    Bump b;
    const size_t e = (size_t)n * g.elems;
    o_g16 = b.take(e * 4); o_ss = b.take((size_t)n * nblk * 4); o_norm = b.take((size_t)n * 4);
    o_xf[0] = b.take(e * 4); o_xf[1] = b.take(e * 4); o_xb[0] = b.take(e * 4); o_xb[1] = b.take(e * 4);
    o_ab = b.take((size_t)n * r * r * 4); o_bb = b.take((size_t)n * r * r * 4); o_ca = b.take((size_t)n * r * r * 4);
    bytes = b.off + 256;
  }
};
}  // namespace

namespace {
template <typename TN>
int newton_schulz_t(int32_t n, int32_t rows, int32_t cols, const float* gin, float* out, int32_t steps, const float* coeffs,
                    int32_t ns_mode, void* workspace, hipStream_t s) {
  const int plain_bf16 = ns_mode == LACT_NS_PLAIN_BF16;
  NsPlan P;
  P.build(n, rows, cols);
  char* ws = align256(workspace);
  // MatGeom treats index 0 as [dh, d] = [rows, cols]; launch with grid.y = n so z / nb == 0 throughout.
  MomentumPrepParams mp;
  memset(&mp, 0, sizeof(mp));
  mp.g = P.g; mp.dw = Partials{gin, 1, 0}; mp.d_out = reinterpret_cast<float*>(ws + P.o_xf[1]);
  mp.g16 = ws + P.o_g16; mp.ss_part = reinterpret_cast<float*>(ws + P.o_ss);
  // partial is indexed [s][3*nb][elems] with z < nb: the layout of gin ([n][elems]) matches for s = 0
  LACT_LAUNCH("k_momentum_prep", "k_momentum_prep", 0.0, (k_momentum_prep<TN>), dim3(P.nblk, n), dim3(256), s, mp);
  NsScaleParams sp;
  memset(&sp, 0, sizeof(sp));
  sp.g = P.g; sp.g16 = mp.g16; sp.ss_part = mp.ss_part; sp.nparts = P.nblk; sp.norms = reinterpret_cast<float*>(ws + P.o_norm);
  sp.xf = reinterpret_cast<float*>(ws + P.o_xf[0]); sp.xb = ws + P.o_xb[0];
  sp.u = steps == 0 ? out : nullptr; sp.plain_bf16 = plain_bf16;
  LACT_LAUNCH("k_ns_scale", "k_ns_scale", 0.0, (k_ns_scale<TN>), dim3(P.nblk, n), dim3(256), s, sp);
  for (int it = 0; it < steps; ++it) {
    const bool last = it + 1 == steps;
    NsIter I;
    I.n = n; I.r = P.r; I.c = P.c; I.nb_for_mask = n; I.mask = P.g.tall(0) ? 1 : 0; I.plain = plain_bf16;
    I.ca = coeffs[3 * it]; I.cb = coeffs[3 * it + 1]; I.cc = coeffs[3 * it + 2];
    I.xf_in = reinterpret_cast<float*>(ws + P.o_xf[it & 1]);
    I.xb_in = ws + P.o_xb[it & 1];
    I.ab = ws + P.o_ab; I.bb = ws + P.o_bb; I.cab = ws + P.o_ca;
    I.xf_out = last ? nullptr : reinterpret_cast<float*>(ws + P.o_xf[(it + 1) & 1]);
    I.xb_out = last ? nullptr : ws + P.o_xb[(it + 1) & 1];
    I.u_out = last ? out : nullptr;
    ns_iteration<TN>(I, s);
  }
  LACT_CHECK_LAUNCH();
  return 0;
}
}  // namespace


// ---- backward of the standalone Newton-Schulz: recomputes the iterates, then walks them backwards ------------
namespace {
struct NsBwdPlan {
  NsPlan f;
  size_t o_xb, o_ab, o_bb, o_gxf[2], o_gxb[2], o_sg, o_gas, o_dot, bytes;
  void build(int n, int rows, int cols, int steps) {
    f.build(n, rows, cols);
    Bump b;
    b.off = f.bytes;
    const size_t e = (size_t)n * f.g.elems, sq = (size_t)n * f.r * f.r, S = (size_t)std::max(1, steps);
    o_xb = b.take(S * e * 4); o_ab = b.take(S * sq * 4); o_bb = b.take(S * sq * 4);
    for (int i = 0; i < 2; ++i) { o_gxf[i] = b.take(e * 4); o_gxb[i] = b.take(e * 4); }
    o_sg = b.take(sq * 4); o_gas = b.take(sq * 4); o_dot = b.take((size_t)n * f.nblk * 4);
    bytes = b.off + 256;
  }
};

template <typename TN>
int newton_schulz_bwd_t(int32_t n, int32_t rows, int32_t cols, const float* gin, const float* dout, float* dg, int32_t steps,
                        const float* coeffs, int32_t ns_mode, void* workspace, hipStream_t s) {
  const int plain_bf16 = ns_mode == LACT_NS_PLAIN_BF16;
  NsBwdPlan P;
  P.build(n, rows, cols, steps);
  const NsPlan& F = P.f;
  char* ws = align256(workspace);
  const size_t e = (size_t)n * F.g.elems, sq = (size_t)n * F.r * F.r;
  auto xb = [&](int it) { return reinterpret_cast<TN*>(ws + P.o_xb) + (size_t)it * e; };
  auto ab = [&](int it) { return reinterpret_cast<TN*>(ws + P.o_ab) + (size_t)it * sq; };
  auto bb = [&](int it) { return reinterpret_cast<TN*>(ws + P.o_bb) + (size_t)it * sq; };
  // ---- forward again, keeping X_k, A_k, B_k
  MomentumPrepParams mp;
  memset(&mp, 0, sizeof(mp));
  mp.g = F.g; mp.dw = Partials{gin, 1, 0}; mp.d_out = nullptr;
  mp.g16 = ws + F.o_g16; mp.ss_part = reinterpret_cast<float*>(ws + F.o_ss);
  LACT_LAUNCH("k_momentum_prep", "k_momentum_prep", 0.0, (k_momentum_prep<TN>), dim3(F.nblk, n), dim3(256), s, mp);
  NsScaleParams sp;
  memset(&sp, 0, sizeof(sp));
  sp.g = F.g; sp.g16 = mp.g16; sp.ss_part = mp.ss_part; sp.nparts = F.nblk; sp.norms = reinterpret_cast<float*>(ws + F.o_norm);
  sp.xf = reinterpret_cast<float*>(ws + F.o_xf[0]); sp.xb = xb(0); sp.plain_bf16 = plain_bf16;
  LACT_LAUNCH("k_ns_scale", "k_ns_scale", 0.0, (k_ns_scale<TN>), dim3(F.nblk, n), dim3(256), s, sp);
  for (int it = 0; it + 1 < steps; ++it) {   // the last iterate itself is not needed
    NsIter I;
    I.n = n; I.r = F.r; I.c = F.c; I.nb_for_mask = n; I.mask = 0; I.plain = plain_bf16;
    I.ca = coeffs[3 * it]; I.cb = coeffs[3 * it + 1]; I.cc = coeffs[3 * it + 2];
    I.xf_in = reinterpret_cast<float*>(ws + F.o_xf[it & 1]); I.xb_in = xb(it);
    I.ab = ab(it); I.bb = bb(it); I.cab = ws + F.o_ca;
    I.xf_out = reinterpret_cast<float*>(ws + F.o_xf[(it + 1) & 1]); I.xb_out = xb(it + 1); I.u_out = nullptr;
    ns_iteration<TN>(I, s);
  }
  if (steps > 0) {   // A and B of the last iteration (its X' is the output the caller already has)
    const int it = steps - 1;
    const long long xe = (long long)F.r * F.c, se = (long long)F.r * F.r;
    auto p = row_params<1>();
    set_term(p.t[0], xb(it), F.c, xe, xb(it), F.c, xe, F.c);
    p.M = F.r; p.N = F.r; p.out = ab(it); p.ldo = F.r; p.bso = se;
    p.out2 = ws + F.o_ca; p.alpha2 = coeffs[3 * it + 2];
    launch_row_gemm<TN, true, 1, EPI_STORE>("ns_gram", p, n, s);
    auto q = row_params<1>();
    set_term(q.t[0], ws + F.o_ca, F.r, se, ab(it), F.r, se, F.r);
    q.M = F.r; q.N = F.r; q.out = bb(it); q.ldo = F.r; q.bso = se;
    q.aux = ab(it); q.ldaux = F.r; q.bsaux = se; q.alpha = 1.f; q.beta = coeffs[3 * it + 1];
    launch_row_gemm<TN, true, 1, EPI_AXPBY>("ns_poly", q, n, s);
  }
  // ---- the incoming gradient where Newton-Schulz holds its matrices
  float* gxf[2] = {reinterpret_cast<float*>(ws + P.o_gxf[0]), reinterpret_cast<float*>(ws + P.o_gxf[1])};
  TN* gxb[2] = {reinterpret_cast<TN*>(ws + P.o_gxb[0]), reinterpret_cast<TN*>(ws + P.o_gxb[1])};
  LACT_LAUNCH("k_to_ns_orientation", "k_to_ns_orientation", 0.0, (k_to_ns_orientation<TN>), dim3(F.nblk, n), dim3(256), s, F.g, dout, gxf[0], (void*)gxb[0]);
  TN* sg = reinterpret_cast<TN*>(ws + P.o_sg);
  TN* gas = reinterpret_cast<TN*>(ws + P.o_gas);
  const long long xe = (long long)F.r * F.c, se = (long long)F.r * F.r;
  int bc = 0;
  for (int it = steps - 1; it >= 0; --it) {
    const float ca = coeffs[3 * it], cb = coeffs[3 * it + 1], cc = coeffs[3 * it + 2];
    {  // Sg = G X^T + X G^T
      auto p = row_params<2>();
      set_term(p.t[0], gxb[bc], F.c, xe, xb(it), F.c, xe, F.c);
      set_term(p.t[1], xb(it), F.c, xe, gxb[bc], F.c, xe, F.c);
      p.M = F.r; p.N = F.r; p.out = sg; p.ldo = F.r; p.bso = se;
      launch_row_gemm<TN, true, 2, EPI_STORE>("ns_bwd_sg", p, n, s);
    }
    {  // gA + gA^T = b Sg + c (Sg A + A Sg)
      auto p = row_params<2>();
      set_term(p.t[0], sg, F.r, se, ab(it), F.r, se, F.r);
      set_term(p.t[1], ab(it), F.r, se, sg, F.r, se, F.r);
      p.M = F.r; p.N = F.r; p.out = gas; p.ldo = F.r; p.bso = se;
      p.aux = sg; p.ldaux = F.r; p.bsaux = se; p.alpha = cc; p.beta = cb;
      launch_row_gemm<TN, true, 2, EPI_AXPBY>("ns_bwd_ga", p, n, s);
    }
    {  // gX = a G + B G + (gA + gA^T) X
      auto p = row_params<2>();
      set_term(p.t[0], bb(it), F.r, se, gxb[bc], F.c, xe, F.r);
      set_term(p.t[1], gas, F.r, se, xb(it), F.c, xe, F.r);
      p.M = F.r; p.N = F.c; p.ldo = F.c; p.bso = xe;
      p.aux = gxf[bc]; p.ldaux = F.c; p.bsaux = xe; p.alpha = 1.f; p.beta = ca;
      p.out = gxf[bc ^ 1]; p.out_c = gxb[bc ^ 1];
      launch_row_gemm<TN, false, 2, EPI_AXPBY_F32_DUAL>("ns_bwd_gx", p, n, s);
    }
    bc ^= 1;
  }
  // ---- backward of X0 = G16 / (|G16| + 1e-7) and of the cast
  NsDotParams dp;
  dp.g = F.g; dp.gx0 = gxf[bc]; dp.g16 = ws + F.o_g16; dp.dot_part = reinterpret_cast<float*>(ws + P.o_dot);
  LACT_LAUNCH("k_ns_bwd_dot", "k_ns_bwd_dot", 0.0, (k_ns_bwd_dot<TN>), dim3(F.nblk, n), dim3(256), s, dp);
  GradPrepParams gp;
  memset(&gp, 0, sizeof(gp));
  gp.g = F.g; gp.gx0 = gxf[bc]; gp.g16 = ws + F.o_g16; gp.norms = reinterpret_cast<float*>(ws + F.o_norm);
  gp.dot_part = dp.dot_part; gp.nparts = F.nblk; gp.gc = dg;
  LACT_LAUNCH("k_grad_prep", "k_grad_prep", 0.0, (k_grad_prep<float, TN>), dim3(F.nblk, n), dim3(256), s, gp);
  LACT_CHECK_LAUNCH();
  return 0;
}
}  // namespace

// ---- Newton-Schulz without a caller workspace: the workspace is a fixed array in device memory -------------
// Every GPU the library runs on holds its own copy of the array (at its own address) until the process ends.
// In host code the array's name is only a handle for hipGetSymbolAddress; the address it returns for the current
// device is what kernels and copies get.
static __device__ __align__(256) unsigned char scratch[LACT_NS_STATIC_WORKSPACE_BYTES];
namespace {
std::mutex g_static_ws_mutex;
void* g_static_ws[64] = {};   // per device: address of `scratch` there
// Address of the static workspace on the current device (looked up once per device), or null with the error set.
void* static_workspace() {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= 64) {
    fail("static workspace: no current device (or device index beyond 63)");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_static_ws_mutex);
  if (!g_static_ws[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      fail(std::string("static workspace: hipGetSymbolAddress failed: ") + hipGetErrorString(e));
      return nullptr;
    }
    g_static_ws[dev] = ptr;
  }
  return g_static_ws[dev];
}
}  // namespace

extern "C" {

const char* lact_last_error(void) { return g_err.c_str(); }
int lact_version(void) { return 1; }

int lact_set_option(int32_t option, int32_t value) {
  std::lock_guard<std::mutex> lock(g_enqueue_mutex);
  if (option == LACT_OPT_NS_BARRIER_SPIN_LIMIT) {
    const long long was = g_ns_spin_limit;
    g_ns_spin_limit = value > 0 ? value : NS_FUSED_SPIN_LIMIT;
    return (int)std::min<long long>(was, 0x7fffffff);
  }
  if (option == LACT_OPT_KEEP_PREACTIVATIONS) {
    const int was = g_keep_pre;
    g_keep_pre = value < 0 ? -1 : (value != 0);
    return was;
  }
  if (option == LACT_OPT_PERSISTENT_TILES) {
    const int was = g_persist;
    g_persist = value;
    return was;
  }
  if (option == LACT_OPT_STREAM_OVERLAP) {
    const int was = g_overlap;
    g_overlap = value > 1 ? 2 : (value != 0);
    return was;
  }
  bool* flag = option == LACT_OPT_FUSED_NEWTON_SCHULZ ? &g_fused_ns : nullptr;
  if (!flag) return fail("lact_set_option: unknown option");
  const int was = *flag ? 1 : 0;
  *flag = value != 0;
  return was;
}

// ---- layer pre- and post-processing -----------------------------------------------------------------
namespace {
int layer_geom(int32_t B, int32_t L, int32_t H, int32_t hd, LayerGeom* g) {
  if (B <= 0 || L <= 0 || H <= 0 || hd <= 0) return fail("layer: B, L, H, hd must be positive");
  if (hd % 4 || hd > LAYER_HD_MAX) return fail("layer: head dim must be a multiple of 4 and at most 1024");
  g->B = B; g->L = L; g->H = H; g->hd = hd;
  return 0;
}
}  // namespace

}  // extern "C"
namespace {
// Calls f(G, NV) for the lanes and chunks (RowLanes) that hd fills best; in fp32 with fewer kernels to choose from.
template <typename T, class F>
void layer_lanes(int hd, F f) {
#define LACT_LANES(limit, G, NV) if (hd <= limit) return f(std::integral_constant<int, G>(), std::integral_constant<int, NV>());
  if constexpr (std::is_same<T, uint16_t>::value) {
    LACT_LANES(64, 16, 1) LACT_LANES(96, 8, 3) LACT_LANES(128, 16, 2) LACT_LANES(192, 16, 3) LACT_LANES(384, 32, 3) LACT_LANES(768, 64, 3)
  } else {
    LACT_LANES(128, 16, 2)
  }
  LACT_LANES(512, 32, 4) LACT_LANES(LAYER_HD_MAX, 64, 4)
#undef LACT_LANES
}
int layer_rows_per_wave(int act_dtype, int hd) {
  int n = 1;
  auto rows = [&](auto g, auto) { n = 64 / decltype(g)::value; };
  if (act_dtype == LACT_BF16) layer_lanes<uint16_t>(hd, rows);
  else layer_lanes<float>(hd, rows);
  return n;
}
unsigned layer_row_blocks(int act_dtype, const LayerGeom& g) {
  const long long n = 4LL * layer_rows_per_wave(act_dtype, g.hd);
  return (unsigned)(((long long)g.B * g.L * g.H + n - 1) / n);
}
// (the number of partial rows that the caller asks for knows neither the type nor hd)
unsigned layer_post_bwd_blocks(const LayerGeom& g) { return (unsigned)std::min(((long long)g.B * g.L * g.H + 3) / 4, 1024LL); }
template <typename T, bool BWD, bool ATT>
void launch_layer_pre_t(const char* name, const char* site, LayerPreParams p, int blocks_per_head, hipStream_t s) {
  layer_lanes<T>(p.g.hd, [&](auto g, auto nv) {
    constexpr int G = decltype(g)::value, NV = decltype(nv)::value;
    p.tokens_per_pass = 4 * (64 / G) * blocks_per_head;
    LACT_LAUNCH(name, site, 0.0, (k_layer_pre<T, BWD, ATT, G, NV>), dim3((unsigned)(blocks_per_head * p.g.H)), dim3(256), s, p);
  });
}
template <bool BWD>
int launch_layer_pre(int act_dtype, const LayerPreParams& p, int blocks_per_head, hipStream_t s) {
  const bool att = p.att[0] || p.datt[0];
  const char* name = BWD ? "k_layer_pre_bwd" : "k_layer_pre";
  const char* site = BWD ? "layer_pre_bwd" : "layer_pre";
  if (act_dtype == LACT_BF16) {
    if (att) launch_layer_pre_t<uint16_t, BWD, true>(name, site, p, blocks_per_head, s);
    else launch_layer_pre_t<uint16_t, BWD, false>(name, site, p, blocks_per_head, s);
  } else if (act_dtype == LACT_F32) {
    if (att) launch_layer_pre_t<float, BWD, true>(name, site, p, blocks_per_head, s);
    else launch_layer_pre_t<float, BWD, false>(name, site, p, blocks_per_head, s);
  } else {
    return fail("act_dtype must be LACT_BF16 or LACT_F32");
  }
  return 0;
}
template <typename T, bool BWD>
void launch_layer_post(const LayerPostParams& p, unsigned blocks, hipStream_t s) {
  layer_lanes<T>(p.g.hd, [&](auto g, auto nv) {
    constexpr int G = decltype(g)::value, NV = decltype(nv)::value;
    LACT_LAUNCH(BWD ? "k_layer_post_bwd" : "k_layer_post", BWD ? "layer_post_bwd" : "layer_post", 0.0, (k_layer_post<T, BWD, G, NV>), dim3(blocks), dim3(256), s, p);
  });
}
int layer_token_blocks(int act_dtype, const LayerGeom& g) {   // one pass of every wave
  const long long n = 4LL * layer_rows_per_wave(act_dtype, g.hd);
  return (int)(((long long)g.B * g.L + n - 1) / n);
}
// Rows of partial sums that a caller provides for the backward with parameter gradients, whatever its type and hd: few enough that they
// stay small beside the activations
int layer_pre_attn_rows(const LayerGeom& g) { return (int)std::max(1LL, std::min(((long long)g.B * g.L + 3) / 4, 1024LL / g.H)); }
// Its blocks per head, one row each: as many as are resident at once, by the waves a SIMD that the registers of one, two or three, and four
// chunks a lane leave.  With three waves' worth for all, us at 16384 tokens (fp32 4096): heads of 64 157 / 144, 1024 109 / 90, fp32 384 67.5 / 61.5.
int layer_pre_attn_blocks(int act_dtype, const LayerGeom& g) {
  int waves = 1;
  auto resident = [&](auto, auto nv) { waves = decltype(nv)::value == 1 ? 4 : decltype(nv)::value < 4 ? 3 : 2; };
  if (act_dtype == LACT_BF16) layer_lanes<uint16_t>(g.hd, resident);
  else layer_lanes<float>(g.hd, resident);
  return std::min(layer_pre_attn_rows(g), std::max(1, 256 * waves / g.H));
}
}  // namespace
extern "C" {

int lact_layer_pre_forward(int32_t act_dtype, int32_t B, int32_t L, int32_t H, int32_t hd, int32_t l2norm, const void* qkv,
                           void* q, void* k, void* v, void* stream) {
  LayerPreParams p;
  memset(&p, 0, sizeof(p));
  if (layer_geom(B, L, H, hd, &p.g)) return -1;
  if (check_ptrs({qkv, q, k, v}, "layer pre tensors")) return -1;
  p.l2norm = l2norm; p.qkv = qkv; p.out[0] = q; p.out[1] = k; p.out[2] = v;
  if (launch_layer_pre<false>(act_dtype, p, layer_token_blocks(act_dtype, p.g), reinterpret_cast<hipStream_t>(stream))) return -1;
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_layer_pre_backward(int32_t act_dtype, int32_t B, int32_t L, int32_t H, int32_t hd, int32_t l2norm, const void* qkv,
                            const void* dq, const void* dk, const void* dv, void* dqkv, void* stream) {
  LayerPreParams p;
  memset(&p, 0, sizeof(p));
  if (layer_geom(B, L, H, hd, &p.g)) return -1;
  if (check_ptrs({qkv, dq, dk, dv, dqkv}, "layer pre backward tensors")) return -1;
  p.l2norm = l2norm; p.qkv = qkv; p.dout[0] = dq; p.dout[1] = dk; p.dout[2] = dv; p.dqkv = dqkv;
  if (launch_layer_pre<true>(act_dtype, p, layer_token_blocks(act_dtype, p.g), reinterpret_cast<hipStream_t>(stream))) return -1;
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_layer_pre_attn_forward(int32_t act_dtype, int32_t B, int32_t L, int32_t H, int32_t hd, int32_t l2norm, int32_t round_product,
                                const void* qkv, const float* qk_scale, const float* qk_offset, void* q, void* k, void* v, void* aq,
                                void* ak, void* av, void* stream) {
  LayerPreParams p;
  memset(&p, 0, sizeof(p));
  if (layer_geom(B, L, H, hd, &p.g)) return -1;
  if (check_ptrs({qkv, qk_scale, qk_offset, q, k, v, aq, ak, av}, "layer pre tensors")) return -1;
  p.l2norm = l2norm; p.qkv = qkv; p.out[0] = q; p.out[1] = k; p.out[2] = v;
  p.att[0] = aq; p.att[1] = ak; p.att[2] = av; p.qk_scale = qk_scale; p.qk_offset = qk_offset; p.round_product = round_product;
  if (launch_layer_pre<false>(act_dtype, p, layer_token_blocks(act_dtype, p.g), reinterpret_cast<hipStream_t>(stream))) return -1;
  LACT_CHECK_LAUNCH();
  return 0;
}

int32_t lact_layer_pre_attn_part_rows(int32_t B, int32_t L, int32_t H) {
  LayerGeom g;
  if (layer_geom(B, L, H, 4, &g)) return -1;
  return layer_pre_attn_rows(g);
}

int lact_layer_pre_attn_backward(int32_t act_dtype, int32_t B, int32_t L, int32_t H, int32_t hd, int32_t l2norm, const void* qkv,
                                 const float* qk_scale, const void* dq, const void* dk, const void* dv, const void* daq, const void* dak,
                                 const void* dav, void* dqkv, float* part, float* dqk_scale, float* dqk_offset, void* stream) {
  LayerPreParams p;
  memset(&p, 0, sizeof(p));
  if (layer_geom(B, L, H, hd, &p.g)) return -1;
  if (check_ptrs({qkv, qk_scale, dq, dk, dv, daq, dak, dav, dqkv, part, dqk_scale, dqk_offset}, "layer pre backward tensors")) return -1;
  p.l2norm = l2norm; p.qkv = qkv; p.dout[0] = dq; p.dout[1] = dk; p.dout[2] = dv; p.dqkv = dqkv;
  p.datt[0] = daq; p.datt[1] = dak; p.datt[2] = dav; p.qk_scale = qk_scale; p.part = part;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int rows = layer_pre_attn_blocks(act_dtype, p.g), dim = H * hd;
  if (launch_layer_pre<true>(act_dtype, p, rows, s)) return -1;
  LACT_LAUNCH("k_layer_qk_reduce", "layer_pre_bwd", 0.0, k_layer_qk_reduce, dim3((dim + 63) / 64, 4), dim3(256), s, part, rows, dim, dqk_scale, dqk_offset);
  LACT_CHECK_LAUNCH();
  return 0;
}

// ---- sliding-window attention of the causal layer
}  // extern "C"
namespace {
int window_attn_params(int B, int L, int H, int D, int window, WindowAttnParams* p) {
  memset(p, 0, sizeof(*p));
  if (B <= 0 || L <= 0 || H <= 0 || window <= 0) return fail("B, L, H and window must be positive");
  if (D != 64 && D != 128) return fail("window attention: head size must be 64 or 128");
  if ((long long)B * H > (1 << 20) || (long long)L * H * D > (1LL << 31)) return fail("window attention: sequence or batch too large");
  p->B = B; p->L = L; p->H = H; p->window = std::min(window, L);
  p->scale = 1.0f / sqrtf((float)D);
  return 0;
}
int attn_rows(const void* ptr, int ld, long long bs, int H, int D, const uint16_t** out_ptr, int* out_ld, long long* out_bs) {
  if (!ptr) return fail("null pointer: window attention tensors");
  if (ld % 8 || bs % 8 || ld < H * D || (reinterpret_cast<uintptr_t>(ptr) & 15)) return fail("window attention: rows must be 16-byte aligned and hold H * D elements");
  if (ld > (1 << 24)) return fail("window attention: row stride too large");
  *out_ptr = static_cast<const uint16_t*>(ptr); *out_ld = ld; *out_bs = bs;
  return 0;
}
// Waves per block: 8 (256 rows, two waves per SIMD) once that gives every compute unit a block, else 4.
template <int D, int NW>
void launch_window_attn(int which, WindowAttnParams p, hipStream_t s) {
  p.by_heads = make_udiv(p.B * p.H);
  const dim3 grid(ceil_div(p.L, 32 * NW) * p.B * p.H), block(64 * NW);
  constexpr int SM = attn_lds_bytes<D, NW>(false), SMS = attn_lds_bytes<D, NW>(true);
  LACT_BIG_LDS((k_window_attn_fwd<D, NW>), SM);
  LACT_BIG_LDS((k_window_attn_dq<D, NW>), SM);
  LACT_BIG_LDS((k_window_attn_dkv<D, NW>), SMS);
  const double w = p.window, pairs = (double)p.L * w - w * (w - 1) / 2, f = 2.0 * pairs * D * p.B * p.H;
  if (which == 0) LACT_LAUNCH_SMEM("k_window_attn_fwd", "window_attn", 2 * f, (k_window_attn_fwd<D, NW>), grid, block, SM, s, p);
  if (which == 1) {
    LACT_LAUNCH_SMEM("k_window_attn_dq", "window_attn_bwd", 3 * f, (k_window_attn_dq<D, NW>), grid, block, SM, s, p);
    LACT_LAUNCH_SMEM("k_window_attn_dkv", "window_attn_bwd", 4 * f, (k_window_attn_dkv<D, NW>), grid, block, SMS, s, p);
  }
}
void launch_window_attn(int which, int D, const WindowAttnParams& p, hipStream_t s) {
  const bool wide = (long long)ceil_div(p.L, 256) * p.B * p.H >= 256;
  if (D == 128) wide ? launch_window_attn<128, 8>(which, p, s) : launch_window_attn<128, 4>(which, p, s);
  else wide ? launch_window_attn<64, 8>(which, p, s) : launch_window_attn<64, 4>(which, p, s);
}
}  // namespace
extern "C" {

int lact_window_attention_forward(int32_t B, int32_t L, int32_t H, int32_t D, int32_t window, const void* q, int32_t q_ld, int64_t q_bs,
                                  const void* k, int32_t k_ld, int64_t k_bs, const void* v, int32_t v_ld, int64_t v_bs, void* out,
                                  float* lse, void* stream) {
  WindowAttnParams p;
  if (window_attn_params(B, L, H, D, window, &p)) return -1;
  if (attn_rows(q, q_ld, q_bs, H, D, &p.q, &p.ldq, &p.bsq) || attn_rows(k, k_ld, k_bs, H, D, &p.k, &p.ldk, &p.bsk) ||
      attn_rows(v, v_ld, v_bs, H, D, &p.v, &p.ldv, &p.bsv))
    return -1;
  if (check_ptrs({out, lse}, "window attention outputs")) return -1;
  p.out = static_cast<uint16_t*>(out); p.lse = lse;
  launch_window_attn(0, D, p, reinterpret_cast<hipStream_t>(stream));
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_window_attention_backward(int32_t B, int32_t L, int32_t H, int32_t D, int32_t window, const void* q, int32_t q_ld, int64_t q_bs,
                                   const void* k, int32_t k_ld, int64_t k_bs, const void* v, int32_t v_ld, int64_t v_bs, const void* out,
                                   const float* lse, const void* dout, int32_t do_ld, int64_t do_bs, float* delta, void* dq, void* dk,
                                   void* dv, void* stream) {
  WindowAttnParams p;
  if (window_attn_params(B, L, H, D, window, &p)) return -1;
  if (attn_rows(q, q_ld, q_bs, H, D, &p.q, &p.ldq, &p.bsq) || attn_rows(k, k_ld, k_bs, H, D, &p.k, &p.ldk, &p.bsk) ||
      attn_rows(v, v_ld, v_bs, H, D, &p.v, &p.ldv, &p.bsv) || attn_rows(dout, do_ld, do_bs, H, D, &p.dout, &p.lddo, &p.bsdo))
    return -1;
  if (check_ptrs({out, lse, delta, dq, dk, dv}, "window attention backward tensors")) return -1;
  p.o = static_cast<const uint16_t*>(out); p.lse = const_cast<float*>(lse); p.delta = delta;
  p.dq = static_cast<uint16_t*>(dq); p.dk = static_cast<uint16_t*>(dk); p.dv = static_cast<uint16_t*>(dv);
  launch_window_attn(1, D, p, reinterpret_cast<hipStream_t>(stream));
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_layer_lr_forward(int32_t B, int32_t L, int32_t H, int32_t rates_major, float base_lr_inv, const float* lr_raw, float* lr0, float* lr1,
                          float* lr2, const float* momentum_raw, float* momentum, void* stream) {
  LayerLrParams p;
  memset(&p, 0, sizeof(p));
  if (layer_geom(B, L, H, 4, &p.g)) return -1;
  if (check_ptrs({lr_raw, lr0, lr1, lr2}, "layer lr tensors")) return -1;
  if (momentum_raw && !momentum) return fail("momentum_raw given without momentum output");
  p.rates_major = rates_major != 0;
  p.base_lr_inv = base_lr_inv; p.lr_raw = lr_raw; p.lr[0] = lr0; p.lr[1] = lr1; p.lr[2] = lr2;
  p.mom_raw = momentum_raw; p.mom = momentum;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const long long n = (long long)B * L * H;
  LACT_LAUNCH("k_layer_lr", "layer_lr", 0.0, (k_layer_lr<false>), dim3((unsigned)((n + 255) / 256)), dim3(256), s, p);
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_layer_lr_backward(int32_t B, int32_t L, int32_t H, int32_t rates_major, float base_lr_inv, const float* lr_raw, const float* dlr0,
                           const float* dlr1, const float* dlr2, float* dlr_raw, const float* momentum_raw,
                           const float* dmomentum, float* dmomentum_raw, void* stream) {
  LayerLrParams p;
  memset(&p, 0, sizeof(p));
  if (layer_geom(B, L, H, 4, &p.g)) return -1;
  if (check_ptrs({lr_raw, dlr_raw}, "layer lr backward tensors")) return -1;
  if (momentum_raw && !dmomentum_raw) return fail("momentum_raw given without dmomentum_raw output");
  p.rates_major = rates_major != 0;
  p.base_lr_inv = base_lr_inv; p.lr_raw = lr_raw; p.dlr[0] = dlr0; p.dlr[1] = dlr1; p.dlr[2] = dlr2; p.dlr_raw = dlr_raw;
  p.mom_raw = momentum_raw; p.dmom = dmomentum; p.dmom_raw = dmomentum_raw;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const long long n = (long long)B * L * H;
  LACT_LAUNCH("k_layer_lr_bwd", "layer_lr_bwd", 0.0, (k_layer_lr<true>), dim3((unsigned)((n + 255) / 256)), dim3(256), s, p);
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_layer_post_add_forward(int32_t act_dtype, int32_t B, int32_t L, int32_t H, int32_t hd, int32_t use_norm, float eps,
                            const void* o, const float* norm_weight, const void* gate_raw, const void* add, void* y, void* stream) {
  LayerPostParams p;
  memset(&p, 0, sizeof(p));
  if (layer_geom(B, L, H, hd, &p.g)) return -1;
  if (check_ptrs({o, y}, "layer post tensors")) return -1;
  p.eps = eps; p.use_norm = use_norm; p.o = o; p.w = norm_weight; p.gate_raw = gate_raw; p.add = add; p.y = y;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (act_dtype == LACT_BF16) launch_layer_post<uint16_t, false>(p, std::min(layer_row_blocks(act_dtype, p.g), 2048u), s);
  else if (act_dtype == LACT_F32) launch_layer_post<float, false>(p, std::min(layer_row_blocks(act_dtype, p.g), 2048u), s);
  else return fail("act_dtype must be LACT_BF16 or LACT_F32");
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_layer_post_forward(int32_t act_dtype, int32_t B, int32_t L, int32_t H, int32_t hd, int32_t use_norm, float eps,
                            const void* o, const float* norm_weight, const void* gate_raw, void* y, void* stream) {
  return lact_layer_post_add_forward(act_dtype, B, L, H, hd, use_norm, eps, o, norm_weight, gate_raw, nullptr, y, stream);
}

int32_t lact_layer_post_dw_rows(int32_t B, int32_t L, int32_t H) {
  LayerGeom g;
  if (layer_geom(B, L, H, 4, &g)) return -1;
  return (int32_t)layer_post_bwd_blocks(g);
}

int lact_layer_post_backward(int32_t act_dtype, int32_t B, int32_t L, int32_t H, int32_t hd, int32_t use_norm, float eps,
                             const void* o, const float* norm_weight, const void* gate_raw, const void* dy, void* d_o,
                             void* dgate_raw, float* dw_part, void* stream) {
  LayerPostParams p;
  memset(&p, 0, sizeof(p));
  if (layer_geom(B, L, H, hd, &p.g)) return -1;
  if (check_ptrs({o, dy, d_o}, "layer post backward tensors")) return -1;
  if (gate_raw && !dgate_raw) return fail("gate_raw given without dgate_raw output");
  p.eps = eps; p.use_norm = use_norm; p.o = o; p.w = norm_weight; p.gate_raw = gate_raw;
  p.dy = dy; p.d_o = d_o; p.dgate_raw = dgate_raw; p.dw_part = use_norm ? dw_part : nullptr;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (act_dtype == LACT_BF16) launch_layer_post<uint16_t, true>(p, layer_post_bwd_blocks(p.g), s);
  else if (act_dtype == LACT_F32) launch_layer_post<float, true>(p, layer_post_bwd_blocks(p.g), s);
  else return fail("act_dtype must be LACT_BF16 or LACT_F32");
  LACT_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
namespace {
// ---- weight gradient of a linear map: dw[M, N] = dy[T, M]^T x[T, N] on the token reduction's kernel ---------------------
struct WeightGradPlan {
  bool big;
  int tiles;
  Split sp;
  size_t bytes;
};
// 192 x 192 tiles where they divide the matrix and are enough of them, else 128 x 128 (768 x 768 from 7500 tokens: 16 tiles of
// 192 leave the split to fill the chip, at a read and a write of a partial sum per 576 tokens).
int weight_grad_plan(int T, int M, int N, WeightGradPlan* w) {
  if (T < 64 || M <= 0 || N <= 0 || M % 8 || N % 8) return fail("weight gradient: 64 tokens or more, features multiples of 8");
  if (M > MAX_ROW_STRIDE || N > MAX_ROW_STRIDE) return fail("row stride too large");
  w->big = M % TS_NS::BM == 0 && N % TS_NS::BN == 0 && (M / TS_NS::BM) * (N / TS_NS::BN) >= 48;
  const int bm = w->big ? TS_NS::BM : TS_SQ::BM, bn = w->big ? TS_NS::BN : TS_SQ::BN;
  w->tiles = ceil_div(M, bm) * ceil_div(N, bn);
  w->sp = choose_split(T, w->tiles, Plan::MAX_SPLITS, 1024);
  w->bytes = w->sp.n > 1 ? (size_t)w->sp.n * M * N * 4 : 0;
  return 0;
}
template <class TS>
void launch_weight_grad(const WeightGradParams& p, double flops, hipStream_t s) {
  constexpr int SM = cmax(DmaSmem<TS, 1, row_stages<TS>()>::BYTES, StageTile<TS, 4>::BYTES);
  LACT_BIG_LDS(k_weight_grad_dma<TS>, SM);
  LACT_LAUNCH_SMEM("k_weight_grad_dma", "weight_grad", flops, (k_weight_grad_dma<TS>), dim3(p.map.grid()), dim3(DMA_THREADS), SM, s, p);
}

// ---- small projections of the layer input -------------------------------------------------------------
constexpr int LAYER_IN_MAX_LR = 24, LAYER_IN_MAX_B16 = 16;   // outputs of the fp32 map and of the bf16 maps together
int layer_in_check(LayerInParams& p, long long rows, int dim) {
  if (rows <= 0 || dim <= 0 || dim % 4) return fail("layer input: rows must be positive, channels a multiple of 4");
  if (p.lr.n < 0 || p.lr.n > LAYER_IN_MAX_LR || p.mom.n < 0 || p.gate.n < 0 || p.mom.n + p.gate.n > LAYER_IN_MAX_B16)
    return fail("layer input: too many outputs");
  if ((p.lr.n && !p.lr.w) || (p.mom.n && !p.mom.w) || (p.gate.n && !p.gate.w)) return fail("null pointer: layer input weights");
  p.rows = rows; p.dim = dim;
  return 0;
}
// The kernels are made for numbers of outputs in fours; a launch takes the next larger one.
int layer_in_nl(const LayerInParams& p) { const int n = (p.lr.n + 3) / 4; return n <= 2 ? 2 : n <= 4 ? n : 6; }
int layer_in_nb(const LayerInParams& p) { const int n = (p.mom.n + p.gate.n + 3) / 4; return n == 0 ? 0 : n <= 2 ? 2 : 4; }
template <int NL, class F>
void layer_in_with_nb(const LayerInParams& p, F f) {
  const int nb = layer_in_nb(p);
  if (nb == 0) f(std::integral_constant<int, NL>(), std::integral_constant<int, 0>());
  else if (nb == 2) f(std::integral_constant<int, NL>(), std::integral_constant<int, 2>());
  else f(std::integral_constant<int, NL>(), std::integral_constant<int, 4>());
}
template <class F>
void layer_in_dispatch(const LayerInParams& p, F f) {
  const int nl = layer_in_nl(p);
  if (nl == 2) layer_in_with_nb<2>(p, f);
  else if (nl == 3) layer_in_with_nb<3>(p, f);
  else if (nl == 4) layer_in_with_nb<4>(p, f);
  else layer_in_with_nb<6>(p, f);
}
// Tokens of a wave in the weight gradients: half as many where the chip would otherwise have fewer than two blocks per unit
// (7500 tokens of 768 channels, 24 outputs: 35 us with 32, 18.6 with 16; more partial sums cost more than they bring at 16384
// tokens of 1536).
int layer_in_dw_tok(long long rows, int dim) { return (rows + 4 * LAYER_IN_DWTOK - 1) / (4 * LAYER_IN_DWTOK) * ceil_div(dim, 256) >= 512 ? LAYER_IN_DWTOK : LAYER_IN_DWTOK / 2; }
int layer_in_parts(long long rows, int dim) { const int n = 4 * layer_in_dw_tok(rows, dim); return (int)((rows + n - 1) / n); }
size_t layer_in_floats(const LayerInParams& p, long long rows, int dim) {
  const int no = 4 * (layer_in_nl(p) + layer_in_nb(p));
  return (size_t)layer_in_parts(rows, dim) * no * (dim + 4);
}
LayerInParams layer_in_maps(const float* wl, int nl, const float* wm, int nm, const float* wg, int ng) {
  LayerInParams p;
  memset(&p, 0, sizeof(p));
  p.lr = LayerInMap{wl, nullptr, nl}; p.mom = LayerInMap{wm, nullptr, nm}; p.gate = LayerInMap{wg, nullptr, ng};
  return p;
}
}  // namespace
extern "C" {

int lact_layer_sum_rows(int32_t rows, int32_t dim, const float* part, float* out, void* stream) {
  if (rows <= 0 || dim <= 0) return fail("sum of rows: rows and columns must be positive");
  if (check_ptrs({part, out}, "sum of rows")) return -1;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  LACT_LAUNCH("k_layer_sum_rows", "layer_sum_rows", 0.0, k_layer_sum_rows, dim3(ceil_div(dim, 64)), dim3(1024), s, part, rows, dim, out);
  LACT_CHECK_LAUNCH();
  return 0;
}

size_t lact_weight_grad_workspace_bytes(int32_t T, int32_t M, int32_t N) {
  WeightGradPlan w;
  return weight_grad_plan(T, M, N, &w) ? 0 : w.bytes;
}

int lact_weight_grad(int32_t T, int32_t M, int32_t N, const void* dy, int32_t dy_ld, const void* x, int32_t x_ld, float* dw,
                     void* workspace, void* stream) {
  WeightGradPlan w;
  if (weight_grad_plan(T, M, N, &w)) return -1;
  if (check_ptrs({dy, x, dw}, "weight gradient tensors")) return -1;
  if (dy_ld < M || x_ld < N || dy_ld % 8 || x_ld % 8 || dy_ld > MAX_ROW_STRIDE || x_ld > MAX_ROW_STRIDE) return fail("weight gradient: row strides");
  if (w.bytes && !workspace) return fail("null pointer: weight gradient workspace");
  WeightGradParams p;
  memset(&p, 0, sizeof(p));
  p.dy = static_cast<const uint16_t*>(dy); p.ldy = dy_ld;
  p.x = static_cast<const uint16_t*>(x); p.ldx = x_ld;
  p.T = T; p.M = M; p.N = N; p.split_len = w.sp.len;
  p.out = w.sp.n == 1 ? dw : static_cast<float*>(workspace);
  p.map = make_tile_map(ceil_div(M, w.big ? TS_NS::BM : TS_SQ::BM), ceil_div(N, w.big ? TS_NS::BN : TS_SQ::BN), w.sp.n);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const double flops = 2.0 * T * M * N;
  if (w.big) launch_weight_grad<TS_NS>(p, flops, s);
  else launch_weight_grad<TS_SQ>(p, flops, s);
  if (w.sp.n > 1) {
    const long long n = (long long)M * N;
    LACT_LAUNCH("k_reduce_partials", "weight_grad", 0.0, k_reduce_partials, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), s, dw, nullptr, 1.f, p.out, w.sp.n, n);
  }
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_layer_in_forward(int64_t rows, int32_t dim, const float* x, const float* mom_w, const float* mom_b, int32_t mom_n,
                          const float* gate_w, const float* gate_b, int32_t gate_n, void* xb, float* mom_raw, void* gate_raw, void* stream) {
  LayerInParams p = layer_in_maps(nullptr, 0, mom_w, mom_n, gate_w, gate_n);
  if (layer_in_check(p, rows, dim)) return -1;
  if (mom_n + gate_n == 0) return fail("layer input: no outputs");
  if (check_ptrs({x, xb}, "layer input tensors")) return -1;
  if ((mom_n && !mom_raw) || (gate_n && !gate_raw)) return fail("null pointer: layer input outputs");
  p.mom.bias = mom_b; p.gate.bias = gate_b;
  p.x = x; p.xb = static_cast<uint16_t*>(xb); p.mom_raw = mom_raw; p.gate_raw = static_cast<uint16_t*>(gate_raw);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)((rows + 4 * LAYER_IN_TOK - 1) / (4 * LAYER_IN_TOK)));
  if (layer_in_nb(p) == 2) LACT_LAUNCH("k_layer_in", "layer_in", 0.0, (k_layer_in<2>), grid, dim3(256), s, p);
  else LACT_LAUNCH("k_layer_in", "layer_in", 0.0, (k_layer_in<4>), grid, dim3(256), s, p);
  LACT_CHECK_LAUNCH();
  return 0;
}

size_t lact_layer_in_backward_workspace_bytes(int64_t rows, int32_t dim, int32_t lr_n, int32_t mom_n, int32_t gate_n) {
  const LayerInParams p = layer_in_maps(nullptr, lr_n, nullptr, mom_n, nullptr, gate_n);
  return layer_in_floats(p, rows, dim) * 4;
}

int lact_layer_in_backward(int64_t rows, int32_t dim, const float* x, const float* lr_w, int32_t lr_n, const float* mom_w, int32_t mom_n,
                           const float* gate_w, int32_t gate_n, const float* dlr_raw, const float* dmom_raw, const void* dgate_raw,
                           const void* dxq, float* dx, float* dlr_w, float* dlr_b, float* dmom_w, float* dmom_b, float* dgate_w,
                           float* dgate_b, void* workspace, void* stream) {
  LayerInParams p = layer_in_maps(lr_w, lr_n, mom_w, mom_n, gate_w, gate_n);
  if (layer_in_check(p, rows, dim)) return -1;
  if (check_ptrs({x}, "layer input tensors")) return -1;
  if (dx && !dxq) return fail("null pointer: layer input gradient");
  p.x = x; p.dlr = dlr_raw; p.dmom = dmom_raw; p.dgate = static_cast<const uint16_t*>(dgate_raw);
  p.dxq = static_cast<const uint16_t*>(dxq); p.dx = dx;
  p.dw[0] = dlr_w; p.dw[1] = dmom_w; p.dw[2] = dgate_w; p.db[0] = dlr_b; p.db[1] = dmom_b; p.db[2] = dgate_b;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int chunks = ceil_div(dim, 256);
  if (dx) {
    int w = 4;                       // waves of a block: as few idle ones as possible
    for (int i = 3; i >= 2; --i)
      if (ceil_div(chunks, i) * i < ceil_div(chunks, w) * w) w = i;
    if (chunks == 1) w = 1;
    const dim3 grid((unsigned)((rows + LAYER_IN_DXTOK - 1) / LAYER_IN_DXTOK), ceil_div(chunks, w));
    layer_in_dispatch(p, [&](auto nl, auto nb) {
    constexpr int NL = decltype(nl)::value, NB = decltype(nb)::value;
    LACT_LAUNCH("k_layer_in_dx", "layer_in_bwd", 0.0, (k_layer_in_dx<NL, NB>), grid, dim3(64 * w), s, p);
  });
  }
  bool any = false;
  for (int i = 0; i < 3; ++i) any = any || p.dw[i] || p.db[i];
  if (any) {
    if (!workspace) return fail("null pointer: layer input workspace");
    const int no = 4 * (layer_in_nl(p) + layer_in_nb(p));
    p.parts = layer_in_parts(rows, dim);
    p.dw_tok = layer_in_dw_tok(rows, dim);
    p.part = static_cast<float*>(workspace);
    p.bpart = p.part + (size_t)p.parts * no * dim;
    layer_in_dispatch(p, [&](auto nl, auto nb) {
    constexpr int NL = decltype(nl)::value, NB = decltype(nb)::value;
    LACT_LAUNCH("k_layer_in_dw", "layer_in_bwd", 0.0, (k_layer_in_dw<NL, NB>), dim3(p.parts, chunks), dim3(256), s, p);
  });
    layer_in_dispatch(p, [&](auto nl, auto nb) {
    constexpr int NL = decltype(nl)::value, NB = decltype(nb)::value;
    LACT_LAUNCH("k_layer_in_reduce", "layer_in_bwd", 0.0, (k_layer_in_reduce<NL, NB>), dim3(ceil_div(dim, 64), no), dim3(256), s, p);
  });
  }
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_check_async_error(void) {
  unsigned n = 0;
  hipError_t e = hipMemcpyFromSymbol(&n, HIP_SYMBOL(g_async_errors), sizeof(n), 0, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return fail(std::string("lact_check_async_error: ") + hipGetErrorString(e));
  if (n == 0) return 0;
  const unsigned zero = 0;
  (void)hipMemcpyToSymbol(HIP_SYMBOL(g_async_errors), &zero, sizeof(zero), 0, hipMemcpyHostToDevice);
  // Whatever held the compute units may still be there: later calls use the unfused launches, which wait for nobody,
  // until the caller switches the fused kernel on again.
  {
    std::lock_guard<std::mutex> lock(g_enqueue_mutex);
    g_fused_ns = false;
  }
  g_err = std::to_string(n) + " barrier wait(s) of the fused Newton-Schulz kernel timed out on this device since the last check: "
          "the results of those steps are NaN (compute units held by another process or kernel).  "
          "LACT_OPT_FUSED_NEWTON_SCHULZ has been switched off: the calls that follow run three launches per iteration, "
          "same results; switch it on again (and, if the waits are merely slow, raise LACT_OPT_NS_BARRIER_SPIN_LIMIT) "
          "once the device is this process's alone";
  return (int)std::min<unsigned>(n, 0x7fffffffu);
}

// Back-to-back matrix instructions on every SIMD of every compute unit: the kernel of known matrix-pipe occupancy
// (all of it) that scales a matrix-busy counter of `rocprofv3 --pmc`, as a plain copy scales the byte counters.
__global__ __launch_bounds__(256) void k_mfma_calibration(int iters, float* out) {
  f32x16 acc[8];
  for (int i = 0; i < 8; ++i)
    for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
  bf16x8 a, b;
  for (int j = 0; j < 8; ++j) { a[j] = (__bf16)(float)((threadIdx.x + j) & 7); b[j] = (__bf16)(float)((threadIdx.x * 3 + j) & 3); }
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[i], 0, 0, 0);
  }
  float sum = 0.f;
  for (int i = 0; i < 8; ++i)
    for (int j = 0; j < 16; ++j) sum += acc[i][j];
  out[(size_t)blockIdx.x * 256 + threadIdx.x] = sum;
}

int lact_mfma_calibration(int32_t blocks, int32_t iters, float* out, void* stream) {
  if (blocks <= 0 || iters <= 0 || !out) return fail("lact_mfma_calibration: bad arguments");
  hipLaunchKernelGGL(k_mfma_calibration, dim3(blocks), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), iters, out);
  LACT_CHECK_LAUNCH();
  return 0;
}

int lact_profile_enable(int on) {
  g_prof.clear();
  g_prof.on = on != 0;
  return 0;
}

int lact_profile_report(char* buf, size_t cap) {
  if (!buf || cap == 0) return fail("null report buffer");
  hipError_t e = hipDeviceSynchronize();
  if (e != hipSuccess) return fail(std::string("synchronize failed: ") + hipGetErrorString(e));
  struct Agg { std::string kernel, site; int stream; long n = 0; double ms = 0, flops = 0; };
  std::vector<Agg> aggs;
  std::vector<hipStream_t> streams;
  for (auto& r : g_prof.recs) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, r.e0, r.e1) != hipSuccess) continue;
    const int stream = (int)(std::find(streams.begin(), streams.end(), r.stream) - streams.begin());
    if (stream == (int)streams.size()) streams.push_back(r.stream);
    Agg* a = nullptr;
    for (auto& x : aggs)
      if (x.kernel == r.kernel && x.site == r.site && x.stream == stream) a = &x;
    if (!a) {
      aggs.push_back(Agg{r.kernel, r.site, stream});
      a = &aggs.back();
    }
    a->n += 1;
    a->ms += ms;
    a->flops += r.flops;
  }
  std::string out = "[";
  for (size_t i = 0; i < aggs.size(); ++i) {
    char line[512];
    snprintf(line, sizeof(line), "%s{\"kernel\": \"%s\", \"site\": \"%s\", \"stream\": %d, \"launches\": %ld, \"ms\": %.6f, \"flops\": %.6e}",
             i ? ", " : "", aggs[i].kernel.c_str(), aggs[i].site.c_str(), aggs[i].stream, aggs[i].n, aggs[i].ms, aggs[i].flops);
    out += line;
  }
  out += "]";
  g_prof.clear();
  if (out.size() + 1 > cap) return fail("report buffer too small");
  memcpy(buf, out.c_str(), out.size() + 1);
  return 0;
}

int lact_query_sizes(const lact_desc_t* desc, size_t* saved_bytes, size_t* scratch_bytes) {
  Plan P;
  if (P.build(desc)) return -1;
  if (saved_bytes) *saved_bytes = P.saved_bytes;
  if (scratch_bytes) *scratch_bytes = P.scratch_bytes;
  return 0;
}

static int run_forward(const lact_desc_t* desc, int n_weights, const float* w0, const float* w1, const float* w2, const void* q, const void* k,
                       const void* v, const float* lr0, const float* lr1, const float* lr2, const float* momentum, const float* const m_in[3],
                       void* out, float* const w_out[3], float* const m_out[3], void* saved, void* scratch, void* stream);

int lact_forward(const lact_desc_t* desc, const float* w0, const float* w1, const float* w2, const void* q, const void* k,
                 const void* v, const float* lr0, const float* lr1, const float* lr2, const float* momentum, void* out,
                 float* const w_out[3], float* const m_out[3], void* saved, void* scratch, void* stream) {
  return run_forward(desc, 0, w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum, nullptr, out, w_out, m_out, saved, scratch, stream);
}

int lact_forward_shared_weights(const lact_desc_t* desc, int32_t n_weights, const float* w0, const float* w1, const float* w2, const void* q,
                                const void* k, const void* v, const float* lr0, const float* lr1, const float* lr2, const float* momentum,
                                void* out, float* const w_out[3], float* const m_out[3], void* saved, void* scratch, void* stream) {
  if (n_weights < 1) return fail("the number of shared weights must be positive");
  return run_forward(desc, n_weights, w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum, nullptr, out, w_out, m_out, saved, scratch, stream);
}

int lact_forward_from_state(const lact_desc_t* desc, const float* w0, const float* w1, const float* w2, const void* q,
                            const void* k, const void* v, const float* lr0, const float* lr1, const float* lr2,
                            const float* momentum, const float* const m_in[3], void* out, float* const w_out[3],
                            float* const m_out[3], void* saved, void* scratch, void* stream) {
  return run_forward(desc, 0, w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum, m_in, out, w_out, m_out, saved, scratch, stream);
}

static int run_forward(const lact_desc_t* desc, int n_weights, const float* w0, const float* w1, const float* w2, const void* q, const void* k,
                       const void* v, const float* lr0, const float* lr1, const float* lr2, const float* momentum, const float* const m_in[3],
                       void* out, float* const w_out[3], float* const m_out[3], void* saved, void* scratch, void* stream) {
  Plan P;
  if (P.build(desc, n_weights)) return -1;
  if (P.state_in && (!m_in || !m_in[0] || !m_in[1] || !m_in[2])) return fail("momentum_state_in set but a state pointer is null");
  if (!P.state_in && m_in) return fail("momentum state passed without momentum_state_in in the descriptor");
  if (check_ptrs({w0, w1, w2, q, out, saved, scratch}, "forward tensors")) return -1;
  if (P.nupd > 0 && check_ptrs({k, v, lr0, lr1, lr2}, "k, v, lr")) return -1;
  if (P.nupd > 0 && P.momentum && !momentum) return fail("use_momentum set but momentum is null");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  std::lock_guard<std::mutex> lock(g_enqueue_mutex);
#define LACT_FWD(T_, TN_)                                                                                           \
  {                                                                                                                 \
    Runner<T_, TN_> R(P, saved, scratch, s);                                                                        \
    return R.forward(w0, w1, w2, (const T_*)q, (const T_*)k, (const T_*)v, lr0, lr1, lr2, momentum, (T_*)out, w_out, \
                     m_out, m_in);                                                                                  \
  }
  const bool ns32 = P.d.ns_mode == LACT_NS_FP32;
  if (P.bf16 && !ns32) LACT_FWD(uint16_t, uint16_t)
  if (P.bf16 && ns32) LACT_FWD(uint16_t, float)
  if (!ns32) LACT_FWD(float, uint16_t)
  LACT_FWD(float, float)
#undef LACT_FWD
}

static int run_backward(const lact_desc_t* desc, int n_weights, const void* q, const void* k, const void* v, const float* lr0, const float* lr1,
                        const float* lr2, const float* momentum, const void* dout, const float* const dw_final[3], const void* saved,
                        void* scratch, float* dw0, float* dw1, float* dw2, void* dq, void* dk, void* dv, float* dlr0, float* dlr1,
                        float* dlr2, float* dmomentum, void* stream) {
  Plan P;
  if (P.build(desc, n_weights)) return -1;
  if (P.d.forward_only) return fail("the forward ran with forward_only set: nothing was kept for a backward pass");
  if (check_ptrs({q, dout, saved, scratch, dw0, dw1, dw2, dq}, "backward tensors")) return -1;
  if (P.nupd > 0 && check_ptrs({k, v, lr0, lr1, lr2, dk, dv, dlr0, dlr1, dlr2}, "k, v, lr and their gradients")) return -1;
  if (P.nupd > 0 && P.momentum && (!momentum || !dmomentum)) return fail("use_momentum set but momentum or dmomentum is null");
  const int al = P.bf16 ? 8 : 4;
  if (P.d.do_ld % al || P.d.do_bs % al || P.d.do_ld < P.d.d) return fail("dout strides must keep 16-byte alignment");
  if (P.d.do_ld > MAX_ROW_STRIDE) return fail("row stride too large");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  std::lock_guard<std::mutex> lock(g_enqueue_mutex);
#define LACT_BWD(T_, TN_)                                                                                            \
  {                                                                                                                  \
    Runner<T_, TN_> R(P, const_cast<void*>(saved), scratch, s);                                                      \
    return R.backward((const T_*)q, (const T_*)k, (const T_*)v, lr0, lr1, lr2, momentum, (const T_*)dout, dw_final,  \
                      dw0, dw1, dw2, (T_*)dq, (T_*)dk, (T_*)dv, dlr0, dlr1, dlr2, dmomentum);                        \
  }
  const bool ns32 = P.d.ns_mode == LACT_NS_FP32;
  if (P.bf16 && !ns32) LACT_BWD(uint16_t, uint16_t)
  if (P.bf16 && ns32) LACT_BWD(uint16_t, float)
  if (!ns32) LACT_BWD(float, uint16_t)
  LACT_BWD(float, float)
#undef LACT_BWD
}

int lact_backward(const lact_desc_t* desc, const void* q, const void* k, const void* v, const float* lr0, const float* lr1,
                  const float* lr2, const float* momentum, const void* dout, const float* const dw_final[3], const void* saved,
                  void* scratch, float* dw0, float* dw1, float* dw2, void* dq, void* dk, void* dv, float* dlr0, float* dlr1,
                  float* dlr2, float* dmomentum, void* stream) {
  return run_backward(desc, 0, q, k, v, lr0, lr1, lr2, momentum, dout, dw_final, saved, scratch, dw0, dw1, dw2, dq, dk, dv, dlr0, dlr1, dlr2,
                      dmomentum, stream);
}

int lact_backward_shared_weights(const lact_desc_t* desc, int32_t n_weights, const void* q, const void* k, const void* v, const float* lr0,
                                 const float* lr1, const float* lr2, const float* momentum, const void* dout, const float* const dw_final[3],
                                 const void* saved, void* scratch, float* dw0, float* dw1, float* dw2, void* dq, void* dk, void* dv, float* dlr0,
                                 float* dlr1, float* dlr2, float* dmomentum, void* stream) {
  if (n_weights < 1) return fail("the number of shared weights must be positive");
  return run_backward(desc, n_weights, q, k, v, lr0, lr1, lr2, momentum, dout, dw_final, saved, scratch, dw0, dw1, dw2, dq, dk, dv, dlr0, dlr1, dlr2,
                      dmomentum, stream);
}

size_t lact_newton_schulz_workspace_bytes(int32_t n, int32_t rows, int32_t cols, int32_t steps) {
  (void)steps;
  if (n <= 0 || rows <= 0 || cols <= 0) return 0;
  NsPlan P;
  P.build(n, rows, cols);
  return P.bytes;
}

int lact_newton_schulz(int32_t n, int32_t rows, int32_t cols, const float* gin, float* out, int32_t steps, const float* coeffs,
                       int32_t ns_mode, void* workspace, void* stream) {
  if (n <= 0 || rows <= 0 || cols <= 0 || n > 65535) return fail("bad Newton-Schulz shape");
  if (rows % 8 || cols % 8) return fail("rows and cols must be multiples of 8");
  if (steps < 0 || steps > 64 || (steps > 0 && !coeffs)) return fail("bad Newton-Schulz steps");
  if (ns_mode < 0 || ns_mode > 2) return fail("ns_mode must be 0, 1 or 2");
  if (!gin || !out || !workspace) return fail("null pointer: newton_schulz");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (ns_mode == LACT_NS_FP32) return newton_schulz_t<float>(n, rows, cols, gin, out, steps, coeffs, ns_mode, workspace, s);
  return newton_schulz_t<uint16_t>(n, rows, cols, gin, out, steps, coeffs, ns_mode, workspace, s);
}

size_t lact_newton_schulz_backward_workspace_bytes(int32_t n, int32_t rows, int32_t cols, int32_t steps) {
  if (n <= 0 || rows <= 0 || cols <= 0 || steps < 0) return 0;
  NsBwdPlan P;
  P.build(n, rows, cols, steps);
  return P.bytes;
}

int lact_newton_schulz_backward(int32_t n, int32_t rows, int32_t cols, const float* gin, const float* dout, float* dg,
                                int32_t steps, const float* coeffs, int32_t ns_mode, void* workspace, void* stream) {
  if (n <= 0 || rows <= 0 || cols <= 0 || n > 65535) return fail("bad Newton-Schulz shape");
  if (rows % 8 || cols % 8) return fail("rows and cols must be multiples of 8");
  if (steps < 0 || steps > 64 || (steps > 0 && !coeffs)) return fail("bad Newton-Schulz steps");
  if (ns_mode < 0 || ns_mode > 2) return fail("ns_mode must be 0, 1 or 2");
  if (!gin || !dout || !dg || !workspace) return fail("null pointer: newton_schulz_backward");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (ns_mode == LACT_NS_FP32) return newton_schulz_bwd_t<float>(n, rows, cols, gin, dout, dg, steps, coeffs, ns_mode, workspace, s);
  return newton_schulz_bwd_t<uint16_t>(n, rows, cols, gin, dout, dg, steps, coeffs, ns_mode, workspace, s);
}

size_t lact_newton_schulz_static_capacity(void) { return LACT_NS_STATIC_WORKSPACE_BYTES; }

int lact_newton_schulz_static(int32_t n, int32_t rows, int32_t cols, const float* gin, float* out, int32_t steps,
                              const float* coeffs, int32_t ns_mode, void* stream) {
  const size_t need = lact_newton_schulz_workspace_bytes(n, rows, cols, steps);
  if (need == 0) return fail("bad Newton-Schulz shape");
  if (need > LACT_NS_STATIC_WORKSPACE_BYTES)
    return fail("lact_newton_schulz_static: n x rows x cols needs " + std::to_string(need) + " workspace bytes, the static workspace holds " +
                std::to_string((size_t)LACT_NS_STATIC_WORKSPACE_BYTES) + " (use lact_newton_schulz with a caller workspace)");
  void* ws = static_workspace();
  if (!ws) return -1;
  return lact_newton_schulz(n, rows, cols, gin, out, steps, coeffs, ns_mode, ws, stream);
}

}  // extern "C"
