// tsa_team.hip -- the variants of k_team (tsa_team.h) without slicing, long work-list entries; and the choice of the team.
#include "tsa_team.h"

hipError_t tsa_launch_team_full(const TsaLaunch& L, int mode, const TsaKParams& P, uint64_t* rec, const uint64_t* leaf,
                                const uint32_t* fix, int nchains, float beta, uint32_t sweep0, int nsweeps,
                                unsigned long long* stats, const TsaEnergyOut& eo, hipStream_t st, hipEvent_t e0,
                                hipEvent_t e1, const TsaLevels* lv, int* res) {
  return tsa_launch_team_t<false, true>(L, mode, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1,
                                   lv, res);
}

void tsa_team_plan(const TsaKParams& P, int nchains, int ncu, int lds_max, int want, TsaLaunch* L) {
  L->team_fits = L->team_full = 0;
  if (want > 8) want = 0;  // (a plan for the wide kernel: it says nothing here)
  L->team_pre = want != 1 && tsa_team_pre_fits(P, lds_max);
  L->pre_sparse = 2ll * nchains < ncu;
  if (want == 1 || P.par_follow || P.par_band > 0) return;
  // the most LDS any launch of the context asks for: a float mode's cache, the level loop, slice moves
  const bool moves = P.slicing && P.slice_moves > 0;
  const int caches = tsa_team_caches(moves, true);
  if (tsa_team_lds(P.m, P.nint, P.W, P.chain_words, 1, caches, 0).bytes > lds_max - TSA_TEAM_STATIC_LDS) return;
  const int per_cu = (nchains + (ncu > 0 ? ncu : 1) - 1) / (ncu > 0 ? ncu : 1);
  // long entries save a visit two dependent LDS round trips; they may not cost a compute unit a chain
  const int most = tsa_team_lds(P.m, P.nint, P.W, P.chain_words, 1, caches, 1).bytes + TSA_TEAM_STATIC_LDS;
  L->team_full = most <= lds_max && (long long)most * per_cu <= lds_max;
  L->team_fits = 1;
  const auto chains = [&](bool loop, int fixed) {  // that LDS holds; fixed: the launch's static LDS
    return lds_max / (tsa_team_lds(P.m, P.nint, P.W, P.chain_words, 0, tsa_team_caches(moves, loop), L->team_full).bytes + fixed);
  };
  const int one = (((P.m * P.W + 1) & ~1) + L->wpb * L->lds_words) * 8 + 512;  // a workgroup of k_sweep
  L->team_rule = TsaTeamRule{want > 0 ? want : 0, per_cu, P.nint * tsa_team_lanes(P.W, 0) / 64,
                             P.nint * tsa_team_lanes(P.W, 1) / 64, P.nint, moves, chains(false, 2640), chains(true, 3392),
                             lds_max / one * L->wpb, P.W};
}
