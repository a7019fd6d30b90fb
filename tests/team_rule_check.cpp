// Waves per chain of the launches given on stdin, one "asked per_cu units units_float nint moves lds lds_loop lds_one
// words mode kind nsweeps" a line (kind: 0 sweeps, 1 block, 2 loop).
#include <cstdio>
#include "tsa_team_rule.h"

int main() {
  int a, c, u, f, n, m, l0, l1, l2, w, mode, kind, s;
  while (std::scanf("%d %d %d %d %d %d %d %d %d %d %d %d %d", &a, &c, &u, &f, &n, &m, &l0, &l1, &l2, &w, &mode, &kind, &s) == 13)
    std::printf("%d\n", tsa_team_waves(TsaTeamRule{a, c, u, f, n, m != 0, l0, l1, l2, w}, mode, (TsaTeamKind)kind, s));
}
