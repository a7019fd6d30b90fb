// Whether pre-order launches run k_team_pre, one "mode W sparse kind nsweeps" a line (kind: 0 sweeps, 2 loop).
#include <cstdio>
#include "tsa_team_rule.h"

int main() {
  int mode, W, sparse, kind, s;
  while (std::scanf("%d %d %d %d %d", &mode, &W, &sparse, &kind, &s) == 5)
    std::printf("%d\n", tsa_pre_pays(mode, W, sparse != 0, (TsaTeamKind)kind, s));
}
