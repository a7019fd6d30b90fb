// tsa_team.hip -- the variants of k_team (tsa_team.h) without slicing, long work-list entries; and the choice of the team.
#include "tsa_team.h"

hipError_t tsa_launch_team_full(const TsaLaunch& L, int mode, const TsaKParams& P, uint64_t* rec, const uint64_t* leaf,
                                const uint32_t* fix, int nchains, float beta, uint32_t sweep0, int nsweeps,
                                unsigned long long* stats, const TsaEnergyOut& eo, hipStream_t st, hipEvent_t e0,
                                hipEvent_t e1, const TsaLevels* lv, int* res) {
  return tsa_launch_team_t<false, true>(L, mode, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1,
                                   lv, res);
}

// The lines lie where the measured times cross (par order, blocks of levels, 40 levels of one sweep, us):
//   chains  sat100: one wave / team of 2 / 4 / 8    sat60                     sq14 (8 words)
//      72            917 / 698 / 548 / 530          692 / 492 / 468 / 475      917 / 632 / 534 / 507
//    1024           1149 / 1097 / 901 / 1071        801 / 704 / 666 / 820     1298 / 1095 / 953 / 1085
//    2048           1491 / 1564 / 1338 / 1829       983 / 901 / 947 / 1329    1880 / 1694 / 1515 / 1872
//    4096           2413 / 2724 / 2416 / 3427      1482 / 1325 / 1603 / 2482  3425 / 3074 / 2799 / 3604
//    6144           3372 / 3908 / 3546 / 5093      1894 / 1891 / 2319 / 3620
// Eight waves pay while a compute unit has one chain; beyond that four where a tree's nodes (times the lanes of a
// proposal) fill them, else two; from 16 chains per unit on, one wave each hides its latency behind the others'.  The
// float modes' visits are long enough for four waves at any size, and their cost cache is the team's alone (gpu mode,
// sat100, 4608 chains: one wave 16.3 ms, two 12.1, four 10.0).  With slice moves a chain holds a second cost cache, and
// from five chains per unit on two waves keep all of them resident (sat70, 2048 chains: 6.9 ms against 10.2 with four).
void tsa_team_plan(const TsaKParams& P, int nchains, int ncu, int lds_max, int want, TsaLaunch* L) {
  L->team = L->team_float = L->team_full = 0;
  L->team_pre = want != 1 && tsa_team_pre_fits(P, lds_max);
  if (want == 1 || want > 8 || P.par_follow || P.par_band > 0) return;
  // the most LDS any launch of the context asks for: a float mode's cache, the level loop, slice moves
  const bool moves = P.slicing && P.slice_moves > 0;
  const int caches = tsa_team_caches(moves, true);
  if (tsa_team_lds(P.m, P.nint, P.W, P.chain_words, 1, caches, 0).bytes > lds_max - TSA_TEAM_STATIC_LDS) return;
  const int per_cu = (nchains + (ncu > 0 ? ncu : 1) - 1) / (ncu > 0 ? ncu : 1);
  // long entries save a visit two dependent LDS round trips; they may not cost a compute unit a chain
  const int most = tsa_team_lds(P.m, P.nint, P.W, P.chain_words, 1, caches, 1).bytes + TSA_TEAM_STATIC_LDS;
  L->team_full = most <= lds_max && (long long)most * per_cu <= lds_max;
  if (want > 1) {
    L->team = L->team_float = want;
    return;
  }
  const int units = P.nint * (P.W <= 2 ? 1 : P.W / 2) / 64;  // wavefuls of lanes that one proposal per node takes
  L->team = per_cu <= 1 ? 8 : per_cu <= 4 ? 4 : per_cu <= 16 ? (units >= 5 && !moves ? 4 : 2) : 0;
  L->team_float = per_cu <= 1 ? 8 : moves && per_cu > 4 ? 2 : 4;
}
