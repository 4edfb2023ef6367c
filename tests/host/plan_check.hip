// Host-side check of the buffer plan (no GPU needed): a token reduction never writes more partial-sum slots than the buffer of its
// chain holds, whatever the lengths of the program's steps, and none of them is held below what its own length asks for on the side
// chain, whose buffer is sized for exactly its launches; and the partial sums of squares of a reduction that folds the momentum step
// in have a place per tile.
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

int main() {
  int bad = 0, n = 0;
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
