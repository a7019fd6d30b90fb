// tsa_wide_pre_pays / tsa_wide_slice_pays of the lines "slice mode W chains compute_units" on stdin.
#include <cstdio>
#include "tsa_wide_rule.h"

int main() {
  int s, mode, W, n, ncu;
  while (std::scanf("%d %d %d %d %d", &s, &mode, &W, &n, &ncu) == 5)
    std::printf("%d\n", s ? tsa_wide_slice_pays(mode, W, n, ncu) : tsa_wide_pre_pays(mode, W, n, ncu));
}
