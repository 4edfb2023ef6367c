// Host-side check of the buffer plan (no GPU needed): a token reduction never writes more partial-sum slots than the buffer of its
// chain holds, whatever the lengths of the program's steps, and none of them is held below what its own length asks for on the side
// chain, whose buffer is sized for exactly its launches; and the partial sums of squares of a reduction that folds the momentum step
// in have a place per tile; and the ranges of k that are scaled by the rates hold every token that an update reads.
#include <cstdio>
#include <cstring>
#include <vector>
#include "../../lact_amd/csrc/plan.h"

using namespace lact;

static int check(bool bf16, int b, int d, int dh, int rounds, int T_update, int T_apply, bool muon) {
  std::vector<lact_step_t> steps;
  int kv = 0, q = 0;
  for (int i = 0; i < rounds; ++i) {
    steps.push_back(lact_step_t{LACT_UPDATE, kv, kv + T_update, 0});
    steps.push_back(lact_step_t{LACT_APPLY, q, q + T_apply, q});
    kv += T_update; q += T_apply;
  }
  lact_desc_t D;
  memset(&D, 0, sizeof(D));
  std::vector<float> coeffs(15, 1.f);
  D.b = b; D.d = d; D.dh = dh; D.q_len = q; D.kv_len = kv; D.out_len = q; D.act_dtype = bf16 ? LACT_BF16 : LACT_F32;
  D.n_steps = (int)steps.size(); D.steps = steps.data(); D.ns_steps = muon ? 5 : -1; D.ns_coeffs = muon ? coeffs.data() : nullptr;
  D.weight_norm = 1; D.q_ld = D.k_ld = D.v_ld = D.o_ld = D.do_ld = d;
  Plan P;
  if (P.build(&D)) { printf("plan refused: %s\n", g_err.c_str()); return 1; }
  int bad = 0;
  auto expect = [&](bool ok, const char* what, int a, int c) {
    if (!ok) { printf("%s: %d against %d (%s b=%d d=%d dh=%d, %d rounds of %d and %d tokens)\n", what, a, c, bf16 ? "bf16" : "fp32", b, d, dh, rounds, T_update, T_apply); ++bad; }
  };
  for (const auto& g : P.groups) {
    const int T = g.st.end - g.st.start, mats = 3 * b * g.n;
    const int wanted = bf16 && T >= 64 ? choose_split(T, tr_tiles(d, dh) * mats, 16, P.split_min).n : choose_split_async(T, P.tiles * mats, 16).n;
    const int used = P.reduce_split(T, g.n, P.max_splits(true, g.n), P.split_min).n;
    expect(used * g.n <= P.side_slots, "slots of a grouped launch", used * g.n, P.side_slots);
    expect(wanted * g.n <= P.side_slots && used == wanted, "splits of a grouped launch", used, wanted);
  }
  for (int T : {T_update, T_apply})
    for (int min_len : {P.split_min, 1536}) {
      const int used = P.reduce_split(T, 1, P.max_splits(false, 1), min_len).n;
      expect(used <= P.nsplit_max, "slots of a launch of the main chain", used, P.nsplit_max);
    }
  if (bf16 && d <= 128)      // an update of small heads as one kernel
    for (int T : {T_update, T_apply}) {
      const Split sp = choose_update_split(T, b, d, dh, P.max_splits(false, 1));
      expect(sp.n <= P.nsplit_max && (sp.n - 1) * sp.len < T && sp.n * sp.len >= T && sp.len % 128 == 0, "splits of an update in one kernel", sp.n, sp.len);
    }
  expect(P.t_partial_side + (size_t)P.side_slots * P.mat3 * 4 <= P.t_gwside, "end of the side buffer", P.side_slots, 0);
  for (const auto& g : P.groups) {
    const size_t rows = (size_t)g.n * b * (g.st.end - g.st.start) * dh * P.esz;
    expect(P.t_hs[0] + rows <= P.t_hs[1] && P.t_hs[1] + rows <= P.t_hs[2] && P.t_hs[2] + rows <= P.t_hn[0], "rows of a grouped launch", g.n, T_apply);
    for (int i = 0; i < g.n; ++i) expect(P.gw_slot[g.ver + i] == P.gw_slot[g.ver] + i && P.gw_slot[g.ver + i] < P.gw_slots, "gradients of a group", g.ver + i, P.gw_slots);
  }
  const size_t newest = (size_t)b * T_apply * dh * P.esz, update = (size_t)b * T_update * dh * P.esz;
  expect(P.t_h[0] + std::max(newest, update) <= P.t_h[1], "rows of the main chain", T_update, T_apply);
  for (int i = 1; i < 6; ++i) expect(P.t_h[i] + update <= (i < 5 ? P.t_h[i + 1] : P.t_hs[0]), "rows of an update", i, T_update);
  for (int i = 0; i < 3; ++i) expect(P.t_hn[i] + newest <= (i < 2 ? P.t_hn[i + 1] : P.t_partial), "rows of the newest version", i, T_apply);
  if (muon) expect(P.t_ss + (size_t)3 * b * std::max(P.nblk, tr_tiles(d, dh)) * 4 <= P.t_dot, "sums of squares per matrix", std::max(P.nblk, tr_tiles(d, dh)), P.nblk);
  return bad;
}

// Updates of `len` tokens (the last one of `last`), their starts `apart` from one another but for the third, which is `shift` later.
static int check_ranges(int n, int first, int apart, int len, int last, int shift) {
  std::vector<lact_step_t> steps;
  int kv = 0, read = 0;
  for (int i = 0; i < n; ++i) {
    const int start = first + i * apart + (i == 2 ? shift : 0), end = start + (i + 1 == n ? last : len);
    steps.push_back(lact_step_t{LACT_UPDATE, start, end, 0});
    kv = std::max(kv, end);
  }
  steps.push_back(lact_step_t{LACT_APPLY, 0, 8, 0});
  lact_desc_t D;
  memset(&D, 0, sizeof(D));
  D.b = 2; D.d = D.dh = 192; D.q_len = 8; D.kv_len = kv + 5; D.out_len = 8; D.act_dtype = LACT_BF16;
  D.n_steps = (int)steps.size(); D.steps = steps.data(); D.ns_steps = -1; D.weight_norm = 1;
  D.q_ld = D.k_ld = D.v_ld = D.o_ld = D.do_ld = 192;
  Plan P;
  if (P.build(&D)) { printf("plan refused: %s\n", g_err.c_str()); return 1; }
  std::vector<char> scaled(P.kl_end - P.kl_begin, 0);
  for (int z = 0; z < P.kl_ranges; ++z)
    for (int t = z * P.kl_period; t < z * P.kl_period + P.kl_len && t < (int)scaled.size(); ++t) scaled[t] += 1;
  bool ok = true, twice = false;
  for (size_t i = 0; i + 1 < steps.size(); ++i)
    for (int t = steps[i].start; t < steps[i].end; ++t, ++read) ok = ok && scaled[t - P.kl_begin];
  int all = 0;
  for (char c : scaled) { twice = twice || c > 1; all += c; }
  // equally far apart with room between them: no more than each update's, as long as the longest
  const bool spaced = apart > 0 && apart > std::max(len, last) && (shift == 0 || n < 3) && n > 1;
  if (ok && !twice && (P.kl_ranges > 1) == spaced && (!spaced || all <= read + std::max(0, len - last) + (n - 1) * std::max(0, last - len))) return 0;
  printf("scaled ranges: %d updates of %d and %d tokens, %d apart from %d on, the third %d later: %d ranges of %d every %d, %d of %d tokens\n", n, len, last, apart, first, shift,
         P.kl_ranges, P.kl_len, P.kl_period, all, read);
  return 1;
}

int main() {
  int bad = 0, n = 0;
  for (int count : {1, 2, 3, 7})
    for (int first : {0, 16})
      for (int apart : {0, 40, 64, 81})
        for (int len : {40, 64, 100})
          for (int last : {24, 40, 64})
            for (int shift : {0, 8}) {
              if (count == 1 && apart) continue;
              bad += check_ranges(count, first, apart, len, count == 1 ? len : last, shift);
              ++n;
            }
  for (bool bf16 : {false, true})
    for (int b : {1, 2, 5})
      for (int d : {8, 64, 128, 192})
        for (int T_update : {40, 256, 1024, 1100, 2049, 4680})
          for (int T_apply : {24, 64, 1000, 1024, 2048, 3000})
            for (int rounds : {1, 2, 4, 9, 70}) {
              bad += check(bf16, b, d, d == 64 ? 96 : d, rounds, T_update, T_apply, rounds == 4) > 0;
              ++n;
            }
  for (int d : {2176, 4096}) { bad += check(true, 1, d, d, 2, 256, 256, true) > 0; ++n; }   // more tiles than blocks of a pass over the matrix
  printf("%d plans checked, %d bad\n", n, bad);
  return bad ? 1 : 0;
}
