// The ordered check of TsaTreeCheck against the traversal: over every pair of children words of m = 3, and over random
// trees (ids in order, or shuffled) with one reference changed, swapped or out of range.  Prints the counts as JSON.
#include <cstdio>
#include <random>
#include <utility>
#include "tsa_valid.h"

int main() {
  TsaTreeCheck check;
  long long cases = 0, valid = 0, ordered = 0, wrong = 0;
  auto one = [&](const uint32_t* ch, int m) {
    const bool o = check.ordered(ch, m), r = check.reached(ch, m);
    cases++;
    valid += r;
    ordered += o;
    bool falls = true;
    for (int i = 0; i < m - 1; i++) falls &= (int)(ch[i] & 0xFFFFu) < m + i && (int)(ch[i] >> 16) < m + i;
    wrong += o != (r && falls) || check(ch, m) != r;
  };
  uint32_t ch[512];
  for (uint32_t a = 0; a < 6 * 6 * 6 * 6; a++) {  // ids 0..5, 5 out of range
    ch[0] = a % 6 | (a / 6 % 6) << 16;
    ch[1] = a / 36 % 6 | (a / 216) << 16;
    one(ch, 3);
  }
  for (uint32_t x : {0u, 0x10000u, 1u, 0x10001u, 0xFFFF0000u, 0x20001u}) one(&x, 2);
  std::mt19937 rng(5);
  for (int k = 0; k < 20000; k++) {
    const int m = 2 + (int)(rng() % 200);
    std::vector<int> roots, name(2 * m - 1);
    for (int i = 0; i < 2 * m - 1; i++) name[i] = i;
    if (k % 3 == 2)  // internal ids below the root in any order
      for (int i = m; i < 2 * m - 2; i++) std::swap(name[i], name[m + (int)(rng() % (unsigned)(m - 2))]);
    for (int i = 0; i < m; i++) roots.push_back(i);
    for (int i = 0; i < m - 1; i++) {
      uint32_t c[2];
      for (int q = 0; q < 2; q++) {
        const size_t j = rng() % roots.size();
        c[q] = (uint32_t)name[roots[j]];
        roots[j] = roots.back();
        roots.pop_back();
      }
      ch[name[m + i] - m] = c[0] | c[1] << 16;
      roots.push_back(m + i);
    }
    one(ch, m);
    uint32_t& w = ch[rng() % (unsigned)(m - 1)];
    const uint32_t id = rng() % 8 == 0 ? rng() & 0xFFFFu : rng() % (unsigned)(2 * m);
    w = rng() & 1 ? (w & 0xFFFFu) | id << 16 : (w & 0xFFFF0000u) | id;
    one(ch, m);
    std::swap(ch[rng() % (unsigned)(m - 1)], ch[rng() % (unsigned)(m - 1)]);
    one(ch, m);
  }
  std::printf("{\"cases\": %lld, \"valid\": %lld, \"ordered\": %lld, \"wrong\": %lld}\n", cases, valid, ordered, wrong);
}
