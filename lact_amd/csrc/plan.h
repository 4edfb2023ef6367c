// What a call needs: the validated program, its scratch and saved buffers, and the rules by which launches are cut that decide
// their sizes.  Host code only; no GPU call.
#pragma once
#include <algorithm>
#include <string>
#include <utility>
#include <vector>

#include "../../include/lact_hip.h"
#include "gemm_dma_kernels.h"
#include "state_kernels.h"

namespace lact {

inline thread_local std::string g_err;
inline int fail(const std::string& m) {
  g_err = m;
  return -1;
}
inline int g_keep_pre = -1;       // LACT_OPT_KEEP_PREACTIVATIONS: -1 by shape, 0 never, 1 whenever the kernels allow it

template <typename T> using TSG = typename AsyncTile<T>::TS;   // tile of the kernels in gemm_kernels.h

struct Bump {
  size_t off = 0;
  size_t take(size_t bytes) {
    const size_t o = off;
    off += (bytes + 255) & ~size_t(255);
    return o;
  }
};

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

struct Split {
  int n, len;
};
// The split count does not grow with the tokens throughout, since splits end on 64 tokens: choose_split_async cuts 1024 tokens into
// eight, 1100 into six.  max_n: slots the partial-sum buffer holds for this launch; min_len: tokens a split has at least
inline Split choose_split(int tokens, int tiles_total, int max_n, int min_len) {
  // One split once the tiles alone occupy most of the 256 compute units: the partial sums then never exist.
  // Otherwise enough splits for one round of blocks, each over at least min_len tokens: partial sums cost a write and a
  // read, which short splits do not earn back.
  int ns = tiles_total >= 160 ? 1 : std::max(1, 256 / std::max(1, tiles_total));
  ns = std::min(std::min(ns, std::max(1, max_n)), std::max(1, tokens / min_len));
  int len = ceil_div(ceil_div(tokens, ns), 64) * 64;
  return Split{ceil_div(tokens, len), len};
}

// The same for the kernel of gemm_kernels.h, whose tiles are small: two rounds of blocks at most, each over at least 128 tokens.
inline Split choose_split_async(int tokens, int tiles_total, int max_n) {
  int ns = std::max(1, 512 / std::max(1, tiles_total));
  ns = std::min(std::min(ns, std::max(1, max_n)), std::max(1, tokens / 128));
  int len = ceil_div(ceil_div(tokens, ns), 64) * 64;
  return Split{ceil_div(tokens, len), len};
}
// Splits of an update of small heads (k_update_fused): blocks of 32 hidden units and a split of the tokens, one to a compute unit,
// those of a batch entry or of a split on one XCD (TileMap).  The least of rounds of blocks times what a block takes -- 2.2 us a 128
// tokens and 8 to start and to add its waves' sums -- and the partial sums' way through memory.  us of the kernel, 6 x 8192 tokens of 128,
// 256 hidden units: 3 splits 74, 5 44, 11 62; 24 x 2500 of 96: 1 split 50, 2 30, 3 24; 8 x 2048 of 64: 4 splits 11.9, 8 8.5, 16 7.4.
inline Split choose_update_split(int tokens, int nb, int d, int dh, int max_n) {
  Split best{1, ceil_div(tokens, 128) * 128};
  double least = 0;
  for (int n = 1; n <= std::max(1, std::min(max_n, ceil_div(tokens, 128))); ++n) {
    const int len = ceil_div(ceil_div(tokens, n), 128) * 128, used = ceil_div(tokens, len), slices = ceil_div(dh, 32);
    const int per_xcd = nb % 8 == 0 ? nb / 8 * used * slices : ceil_div(nb * used, 8) * slices;
    const double t = ceil_div(per_xcd, 32) * (len / 128 * 2.2 + 8.0) + (double)used * nb * 3 * d * dh * 8 / 4e6;
    if (n == 1 || t < least) { least = t; best = Split{used, len}; }
  }
  return best;
}
template <typename T>
int token_reduce_tiles(int d, int dh) {
  return std::max(ceil_div(dh, TSG<T>::BM) * ceil_div(d, TSG<T>::BN), ceil_div(d, TSG<T>::BM) * ceil_div(dh, TSG<T>::BN));
}

// Tile of the dedicated-loader token reduction: 192 x 192 where it divides the matrices, else 128 x 128.  (128 x 64 where few
// matrices leave the chip idle was measured: a block's K-step takes as long as with the large tile -- it waits for operands
// that another kernel has just written -- and the launch copies more: 12 matrices of 384 x 384, 2048 tokens, 28.7 us in 48
// blocks of 192 x 192, 28.2 us in 216 of 128 x 64, the launch that also holds the dk and dv GEMMs 34 against 42 us.)
inline bool tr_big(int d, int dh) { return d % TS_NS::BM == 0 && dh % TS_NS::BM == 0; }
inline int tr_tiles(int d, int dh) {   // output tiles per matrix
  return tr_big(d, dh) ? (d / TS_NS::BM) * (dh / TS_NS::BN)
                       : std::max(ceil_div(dh, TS_SQ::BM) * ceil_div(d, TS_SQ::BN), ceil_div(d, TS_SQ::BM) * ceil_div(dh, TS_SQ::BN));
}

// One Newton-Schulz launch group: n matrices of one geometry, laid out one after the other.
struct NsBatch {
  int n, r, c;          // matrices, Newton-Schulz orientation [r, c] (r <= c)
  int mask, nb;         // the orthogonalised update of matrix z is written back transposed when bit (z / nb) of mask is set
  int first;            // index of its first matrix among all Newton-Schulz matrices (barrier lines)
  size_t xoff, sqoff;   // element offsets: [r, c]-shaped buffers (and the update in original orientation); [r, r]-shaped buffers
};

// Apply steps of consecutive weight versions, equally long and equally spaced: one launch covers all of them.
struct ApplyGroup {
  lact_step_t st;                  // the first step
  int ver, n;                      // its weight version; number of steps
  int dstart, dout;                // from one step's rows of q, of the output, to the next one's
};

// Largest distance of two rows, in elements: the kernels form a tile's byte offsets from 24-bit products.
constexpr int MAX_ROW_STRIDE = (1 << 23) - 1;

struct Plan {
  lact_desc_t d;
  std::vector<NsBatch> nsb;
  size_t sq_total = 0;    // elements of one [r, r]-shaped buffer over all batches
  std::vector<lact_step_t> steps;
  std::vector<lact_step_t> live;    // the steps that are executed: `steps` without the apply rows a later step overwrites
  std::vector<ApplyGroup> groups;   // the apply steps among them whose version is not the newest
  std::vector<int> gw_slot;         // by version: place of the gradient that its grouped steps leave for the update chain; -1: it has none
  int gw_slots = 0;
  int Tnew = 0;                     // longest apply step on the newest version
  std::vector<float> coeffs;
  MatGeom g;
  int nupd = 0, Tcap = 0, Tupd = 1, S = -1, esz = 2, nsz = 2, r = 0, c = 0, nblk = 1, lr_slots = 1, tiles = 1, nsplit_max = 1, mdot_parts = 1, split_min = 1024, kl_begin = 0, kl_end = 0, side_slots = 1;
  int kl_period = 0, kl_len = 0, kl_ranges = 1;   // of [kl_begin, kl_end) updates read the first kl_len tokens of every kl_period
  double side_work = 0;   // of the grouped apply steps' forward, in operations of bf16
  int nw = 0;       // initial weights and their gradients: matrices of each kind, batch entry i uses i % nw
  bool muon = false, bf16 = true, momentum = false, state_in = false;
  size_t mat3 = 0;  // 3*b*elems
  // saved
  size_t s_n0, s_wf, s_wc, s_main, s_d, s_min, s_mbar, s_u, s_g16, s_norms, s_xb, s_ab, s_bb, saved_bytes;
  // Kept for the backward on the asynchronous-copy path: per update, six token-major arrays [b][T][dh] -- the three
  // lr-scaled hidden-side operands the backward's GEMMs read and the three rounded pre-activations they came from.
  // (The two unscaled operands of the forward's dw0 / dw2 reductions, which scale k instead, are read by the forward's
  // own token reduction only: they live in the call's scratch.)
  // 288 GB of HBM make keeping them cheaper than the three GEMMs that would recompute them.
  bool keep_pre = false;
  std::vector<size_t> s_pre;   // by update index
  std::vector<int> pre_T;
  // scratch
  size_t t_h[6], t_partial, t_lrpart, t_xf[2], t_xbtmp, t_ss, t_dot, t_mdot, t_gwhat[2], t_gwcur, t_gmcarry, t_gc,
      t_gxf[2], t_gxb[2], t_sg, t_gas, t_gn0, t_hs[3], t_hn[3], t_partial_side, t_gwside, t_nssync, t_kl[2], t_ca, scratch_bytes;

  // n_weights: matrices of each kind that the batch entries share, 0: every entry has its own
  int build(const lact_desc_t* desc, int n_weights = 0) {
    if (!desc) return fail("null descriptor");
    d = *desc;
    if (d.b <= 0 || d.d <= 0 || d.dh <= 0) return fail("b, d, dh must be positive");
    if (n_weights < 0 || (n_weights > 0 && d.b % n_weights)) return fail("the number of shared weights must divide b");
    nw = n_weights > 0 ? n_weights : d.b;
    if (d.d % 8 || d.dh % 8) return fail("d and dh must be multiples of 8");
    if (d.act_dtype != LACT_BF16 && d.act_dtype != LACT_F32) return fail("act_dtype must be LACT_BF16 or LACT_F32");
    bf16 = d.act_dtype == LACT_BF16;
    esz = bf16 ? 2 : 4;
    const int al = bf16 ? 8 : 4;
    if (d.q_ld % al || d.k_ld % al || d.v_ld % al || d.o_ld % al || d.q_bs % al || d.k_bs % al || d.v_bs % al ||
        d.o_bs % al)
      return fail("row and batch strides must keep 16-byte alignment");
    if (d.q_ld < d.d || d.k_ld < d.d || d.v_ld < d.d || d.o_ld < d.d) return fail("row stride smaller than d");
    if (std::max(std::max(d.q_ld, d.k_ld), std::max(d.v_ld, d.o_ld)) > MAX_ROW_STRIDE || d.d > MAX_ROW_STRIDE || d.dh > MAX_ROW_STRIDE)
      return fail("row stride too large");
    if (3LL * d.b > 65535) return fail("b too large (3*b must fit a grid dimension)");
    if (d.n_steps <= 0 || !d.steps) return fail("empty program");
    steps.assign(d.steps, d.steps + d.n_steps);
    S = d.ns_steps;
    muon = S >= 0;
    if (S > 0 && !d.ns_coeffs) return fail("ns_coeffs missing");
    if (S > 64) return fail("too many Newton-Schulz steps");
    if (S > 0) coeffs.assign(d.ns_coeffs, d.ns_coeffs + 3 * S);
    momentum = d.use_momentum != 0;
    state_in = d.momentum_state_in != 0;
    if (state_in && (!momentum || !d.forward_only))
      return fail("momentum_state_in needs use_momentum and forward_only (the carried state has no backward pass)");
    if (d.ns_mode < 0 || d.ns_mode > 2) return fail("ns_mode must be 0, 1 or 2");
    nsz = d.ns_mode == LACT_NS_FP32 ? 4 : 2;
    nupd = 0;
    Tcap = 0;
    Tupd = 1;
    for (const auto& s : steps) {
      if (s.kind != LACT_UPDATE && s.kind != LACT_APPLY) return fail("step kind must be LACT_UPDATE or LACT_APPLY");
      if (s.start < 0 || s.end <= s.start) return fail("empty or negative step range");
      if (s.kind == LACT_UPDATE) {
        if (s.end > d.kv_len) return fail("update range exceeds kv_len");
        ++nupd;
        Tupd = std::max(Tupd, s.end - s.start);
      } else {
        if (s.end > d.q_len) return fail("apply range exceeds q_len");
        if (s.out_start < 0 || s.out_start + (s.end - s.start) > d.out_len) return fail("apply output range exceeds out_len");
      }
      Tcap = std::max(Tcap, s.end - s.start);
    }
    // Output rows that a later apply step writes again are dead in the earlier one (the reference's slice
    // assignment lets the later write win, and no gradient reaches the overwritten values): every apply step is
    // cut down to the rows that survive, in the forward and in the backward alike.  What is left never writes a
    // row twice, so the apply steps may run in any order.
    live.clear();
    for (size_t i = 0; i < steps.size(); ++i) {
      const lact_step_t& a = steps[i];
      if (a.kind != LACT_APPLY) { live.push_back(a); continue; }
      std::vector<std::pair<int, int>> keep(1, std::make_pair(a.out_start, a.out_start + (a.end - a.start)));
      for (size_t j = i + 1; j < steps.size() && !keep.empty(); ++j) {
        const lact_step_t& b = steps[j];
        if (b.kind != LACT_APPLY) continue;
        const int b0 = b.out_start, b1 = b.out_start + (b.end - b.start);
        std::vector<std::pair<int, int>> next;
        for (auto& iv : keep) {
          if (b1 <= iv.first || iv.second <= b0) { next.push_back(iv); continue; }
          if (iv.first < b0) next.emplace_back(iv.first, b0);
          if (b1 < iv.second) next.emplace_back(b1, iv.second);
        }
        keep.swap(next);
      }
      for (auto& iv : keep) {
        lact_step_t c = a;
        c.start = a.start + (iv.first - a.out_start);
        c.end = c.start + (iv.second - iv.first);
        c.out_start = iv.first;
        live.push_back(c);
      }
    }
    g.d = d.d;
    g.dh = d.dh;
    g.nb = d.b;
    g.elems = (long long)d.d * d.dh;
    r = std::min(d.d, d.dh);
    c = std::max(d.d, d.dh);
    mat3 = (size_t)3 * d.b * g.elems;
    g.stacked = (muon && d.muon_stacked) ? 1 : 0;
    if (g.stacked && S == 0) return fail("muon_stacked needs at least one Newton-Schulz iteration");
    nsb.clear();
    if (!g.stacked) {
      nsb.push_back(NsBatch{3 * d.b, r, c, (g.tall(0) ? 1 : 0) | (g.tall(1) ? 2 : 0) | (g.tall(2) ? 4 : 0), d.b, 0, 0, 0});
      sq_total = (size_t)3 * d.b * r * r;
    } else {
      const int rs = std::min(2 * d.dh, d.d), cs = std::max(2 * d.dh, d.d);
      nsb.push_back(NsBatch{d.b, rs, cs, 2 * d.dh > d.d ? 1 : 0, d.b, 0, 0, 0});
      nsb.push_back(NsBatch{d.b, r, c, g.tall(1) ? 1 : 0, d.b, d.b, (size_t)2 * d.b * g.elems, (size_t)d.b * rs * rs});
      sq_total = (size_t)d.b * rs * rs + (size_t)d.b * r * r;
    }
    nblk = std::max(1, std::min(256, (int)((g.elems + 2047) / 2048)));
    lr_slots = ceil_div(d.dh, 128) * 4;   // (hidden tiles) x (wave columns) of the widest update-backward tiling
    tiles = bf16 ? token_reduce_tiles<uint16_t>(d.d, d.dh) : token_reduce_tiles<float>(d.d, d.dh);
    // partial-sum slots of the main chain: the larger split count of the two token-reduction kernels at the longest step; a
    // shorter step's launch is held to it (reduce_split).
    // With Newton-Schulz the partial sums are read by a pass of its own, and one split lets the reduction's epilogue do the momentum
    // step; without, the row kernels add them up on the way (12 matrices of 384 x 384, 2048 tokens, us of the reduction and of
    // the renorm that reads it: one split 30.3 + 9.3, two 21.5 + 10.1, four 18.3 + 12.2).
    split_min = muon ? 1536 : 1024;
    nsplit_max = std::max(choose_split_async(Tcap, tiles * 3 * d.b, MAX_SPLITS).n, choose_split(Tcap, tr_tiles(d.d, d.dh) * 3 * d.b, MAX_SPLITS, split_min).n);
    if (bf16 && d.d <= 128) nsplit_max = std::max(nsplit_max, choose_update_split(Tcap, d.b, d.d, d.dh, MAX_SPLITS).n);
    mdot_parts = std::max(std::max(nblk, 256), ceil_div(g.maxrows(), 4));
    build_groups();
    side_slots = 1;
    size_t side_rows = 0;     // rows of the largest group
    for (const ApplyGroup& g : groups) {
      const int T = g.st.end - g.st.start;
      side_slots = std::max(side_slots, g.n * reduce_split(T, g.n, MAX_SPLITS, split_min).n);
      side_rows = std::max(side_rows, (size_t)g.n * T);
    }

    Bump sv;
    s_n0 = sv.take((size_t)3 * d.b * g.maxrows() * 4);
    s_wf = sv.take((size_t)(nupd + 1) * mat3 * 4);
    s_wc = bf16 ? sv.take((size_t)(nupd + 1) * mat3 * 2) : s_wf;
    s_main = d.prenorm ? sv.take((size_t)nupd * mat3 * 4) : 0;
    s_d = sv.take((size_t)nupd * mat3 * 4);
    s_min = state_in ? sv.take(mat3 * 4) : 0;
    s_mbar = sv.take((size_t)std::max(1, nupd) * d.b * 4);
    s_u = muon ? sv.take((size_t)nupd * mat3 * 4) : 0;
    s_g16 = muon ? sv.take((size_t)nupd * mat3 * nsz) : 0;
    s_norms = sv.take((size_t)std::max(1, nupd) * 3 * d.b * 4);
    s_xb = muon ? sv.take((size_t)nupd * std::max(1, S) * mat3 * nsz) : 0;
    const size_t sq3 = sq_total;
    s_ab = muon ? sv.take((size_t)nupd * std::max(1, S) * sq3 * nsz) : 0;
    s_bb = muon ? sv.take((size_t)nupd * std::max(1, S) * sq3 * nsz) : 0;
    // Keep the update's rounded pre-activations and lr-scaled operands for the backward (three GEMM phases there
    // instead of six), or let the backward recompute them?  Recomputing costs K = d of matrix work per tile and saves
    // five token-major arrays of stores in the forward: at d <= 128 (two K-steps) recomputing wins (d = 128, dh = 256,
    // 32760 tokens: 3.61 against 3.70 ms per step), at d = 384 keeping does (1.298 against 1.316 ms; 7.38 against 7.47).
    keep_pre = bf16 && d.d % 64 == 0 && d.dh % 64 == 0 && !d.forward_only && (g_keep_pre < 0 ? d.d > 128 : g_keep_pre != 0);
    s_pre.clear(); pre_T.clear();
    if (keep_pre)
      for (const auto& st : steps)
        if (st.kind == LACT_UPDATE) {
          pre_T.push_back(st.end - st.start);
          s_pre.push_back(sv.take((size_t)6 * d.b * (st.end - st.start) * d.dh * esz));
        }
    saved_bytes = sv.off + 256;

    // What only a backward pass uses is left out of a forward-only call.
    Bump sc;
    const bool bwd = !d.forward_only;
    auto take_bwd = [&](size_t bytes) { return sc.take(bwd ? bytes : 0); };
    // Token-major arrays of the hidden size, the batch entries of a step one after the other: each as long as the steps that use it.
    const size_t row = (size_t)d.b * d.dh * esz;
    for (int i = 0; i < 3; ++i) t_h[i] = sc.take((i == 0 ? std::max(Tupd, Tnew) : Tupd) * row);
    for (int i = 3; i < 6; ++i) t_h[i] = take_bwd(Tupd * row);
    for (int i = 0; i < 3; ++i) t_hs[i] = i == 0 ? sc.take(side_rows * row) : take_bwd(side_rows * row);   // the grouped apply steps', which run beside the update chain
    for (int i = 0; i < 3; ++i) t_hn[i] = take_bwd(Tnew * row);       // those of the newest version
    t_partial = sc.take((size_t)nsplit_max * mat3 * 4);
    t_lrpart = take_bwd((size_t)std::max(1, nupd) * 3 * lr_slots * d.b * Tupd * 4);   // one slot per update: reduced by one launch at the end
    for (int i = 0; i < 2; ++i) t_xf[i] = sc.take(mat3 * 4);
    t_xbtmp = sc.take(mat3 * nsz);
    t_ss = sc.take((size_t)3 * d.b * std::max(nblk, tr_tiles(d.d, d.dh)) * 4);   // per block of a pass over the matrix, or per tile of the reduction that folds the pass in
    t_dot = take_bwd((size_t)3 * d.b * std::max(nblk, 32) * 4);   // partial dots: per chunk of a matrix, or per block of the fused kernel
    t_mdot = take_bwd((size_t)std::max(1, nupd) * 3 * d.b * mdot_parts * 4);   // one slot per update: the momentum gradients are written at the end
    for (int i = 0; i < 2; ++i) t_gwhat[i] = take_bwd(mat3 * 4);
    t_gwcur = take_bwd(mat3 * 4);
    t_gmcarry = take_bwd(mat3 * 4);
    t_gc = take_bwd(mat3 * esz);
    for (int i = 0; i < 2; ++i) t_gxf[i] = take_bwd(mat3 * 4);
    for (int i = 0; i < 2; ++i) t_gxb[i] = take_bwd(mat3 * nsz);
    t_sg = take_bwd(sq3 * nsz);
    t_gas = take_bwd(sq3 * nsz);
    t_gn0 = take_bwd((size_t)3 * d.b * g.maxrows() * 4);
    t_partial_side = take_bwd((size_t)side_slots * mat3 * 4);
    t_gwside = take_bwd((size_t)std::max(1, gw_slots) * mat3 * 4);   // by gw_slot
    t_nssync = sc.take(((size_t)3 * d.b * 32 + 32) * 4);   // per-matrix barrier lines of the fused Newton-Schulz kernel + error word
    // k * lr0, k * lr2 of the tokens [kl_begin, kl_end) that updates read
    kl_begin = d.kv_len; kl_end = 0;
    for (const auto& st : steps)
      if (st.kind == LACT_UPDATE) { kl_begin = std::min(kl_begin, st.start); kl_end = std::max(kl_end, st.end); }
    scale_ranges();
    for (int i = 0; i < 2; ++i) t_kl[i] = sc.take((size_t)d.b * std::max(0, kl_end - kl_begin) * d.d * esz);
    t_ca = muon ? sc.take(sq3 * nsz) : 0;                   // c * A of the current Newton-Schulz iteration
    scratch_bytes = sc.off + 256;
    return 0;
  }
  static constexpr int MAX_SPLITS = 16;
  // bf16, 64 tokens or more: the dedicated-loader kernel, else the one of gemm_kernels.h
  bool reduce_on_dma(int tokens) const { return bf16 && tokens >= 64; }
  // How the token reduction of a launch over `steps` steps of `tokens` tokens each is cut.
  Split reduce_split(int tokens, int steps, int max_n, int min_len) const {
    const int mats = 3 * d.b * steps;
    return reduce_on_dma(tokens) ? choose_split(tokens, tr_tiles(d.d, d.dh) * mats, max_n, min_len) : choose_split_async(tokens, tiles * mats, max_n);
  }
  // Most splits that launch may have: what the partial-sum buffer of its chain holds (every split writes `steps` slots of mat3 elements).
  int max_splits(bool on_side, int steps) const { return std::min(MAX_SPLITS, (on_side ? side_slots : nsplit_max) / steps); }
  // Updates with tokens between them, their starts equally far apart: k is scaled for theirs only.  Everything else is one range.
  void scale_ranges() {
    kl_ranges = 1;
    kl_period = kl_len = std::max(0, kl_end - kl_begin);
    int last = -1, apart = 0, longest = 0, n = 0;
    for (const auto& st : live) {
      if (st.kind != LACT_UPDATE) continue;
      if (n == 1) apart = st.start - last;
      if (n > 0 && (st.start - last != apart || apart <= 0)) return;
      last = st.start;
      longest = std::max(longest, st.end - st.start);
      ++n;
    }
    if (n < 2 || n > 65535 || longest >= apart) return;
    kl_ranges = n; kl_period = apart; kl_len = longest;
  }
  // Groups of as many steps as it takes to give every compute unit a 128 x 128 tile of the hidden stage.  Fewer, fuller launches,
  // and fewer event waits at 12 us of host time each: 8 chunks of 64 rows in fp32 526 -> 480 us, 15 of 192 tiles
  // 2.83 -> 2.79 ms; twice the size gains nothing more and delays the chain, which waits for whole groups (many small chunks with
  // Newton-Schulz: 839 us, 853 with twice the size).
  void build_groups() {
    groups.clear();
    gw_slot.assign(nupd + 1, -1);
    gw_slots = 0;
    Tnew = 0;
    side_work = 0;
    int ver = 0;
    for (const auto& st : live) {
      if (st.kind == LACT_UPDATE) { ++ver; continue; }
      const int T = st.end - st.start;
      if (ver == nupd) { Tnew = std::max(Tnew, T); continue; }
      if (gw_slot[ver] < 0) gw_slot[ver] = gw_slots++;
      side_work += 6.0 * T * d.d * d.dh * d.b * (bf16 ? 1 : 9);      // (fp32 products run at a ninth of the rate)
      const long long tiles1 = (long long)ceil_div(T, 128) * ceil_div(d.dh, 128) * d.b;
      const int limit = (int)std::max(1LL, std::min(std::min(65535LL / (3 * d.b), 64LL), (256 + tiles1 - 1) / tiles1));
      if (!groups.empty()) {
        ApplyGroup& g = groups.back();
        const int ds = st.start - (g.st.start + (g.n - 1) * g.dstart), dout = st.out_start - (g.st.out_start + (g.n - 1) * g.dout);
        // rows of q that two steps share would be two additions to one gradient row
        if (g.n < limit && ver == g.ver + g.n && T == g.st.end - g.st.start && (ds >= T || ds <= -T) && (g.n == 1 || (ds == g.dstart && dout == g.dout))) {
          g.dstart = ds; g.dout = dout;
          ++g.n;
          continue;
        }
      }
      groups.push_back(ApplyGroup{st, ver, 1, 0, 0});
    }
  }
};

}  // namespace lact
