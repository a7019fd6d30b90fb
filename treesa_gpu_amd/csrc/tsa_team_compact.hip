// tsa_team_compact.hip -- the variants of k_team (tsa_team.h) without slicing, short work-list entries.
#include "tsa_team.h"

hipError_t tsa_launch_team_compact(const TsaLaunch& L, int mode, const TsaKParams& P, uint64_t* rec, const uint64_t* leaf,
                                   const uint32_t* fix, int nchains, float beta, uint32_t sweep0, int nsweeps,
                                   unsigned long long* stats, const TsaEnergyOut& eo, hipStream_t st, hipEvent_t e0,
                                   hipEvent_t e1, const TsaLevels* lv, int* res) {
  return tsa_launch_team_t<false, false>(L, mode, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1,
                                   lv, res);
}
