// tsa_wide_rule.h -- whether pre-order sweeps and sliced par sweeps of label sets in HBM run on lane groups
// (tsa_wide_pre.hip, k_wide with SLICE) or one lane per proposal (k_sweep).  Plain C++, also compiled by the CPU tests.
//
// A lane group makes a proposal short, which is what counts while a compute unit has few chains; with many it is the
// work that counts, and of a narrow set most of a group's lanes have no word, while in the float modes all of them
// evaluate the energy.  W: 64-bit words per label set.  Ratios below: one lane's time over the lane groups' (launch and
// energies, MI355X), at 256, 512, 1024, 2048, 4096 chains.
#pragma once

// Pre-order.  tc mode: W = 4 1.49 - 1.01 0.64 0.58, W = 8 2.35 - 1.55 1.15 1.02.  Float modes (gpu): W = 4 0.99 - 0.56 0.38,
// W = 8 1.20 (768 chains: 0.76) 0.59 0.46, W = 16 1.72 (768: 1.06) 0.91 0.63, W = 24 2.23 - 1.27 0.97 0.98, W = 32 2.34 -
// 1.46 1.49 1.72.
static inline bool tsa_wide_pre_pays(int mode, int W, int nchains, int ncu) {
  if (mode == 0) return W >= 8 || nchains <= 4 * ncu;
  return W >= 32 || 5ll * nchains <= (long long)ncu * W;
}

// Par with slice sets.  tc mode: W = 4 1.27 0.75 0.43, W = 6 1.75 1.03 0.62, W = 8 2.21 1.33 (768: 0.99) 0.83 0.72, W = 10
// 2.64 1.62 1.08 1.03 1.09.  gpu mode: W = 4 1.14 0.65 0.36, W = 8 2.17 1.24 (768: 0.89) 0.72, W = 10 2.45 1.38 (768: 1.01)
// 0.84, W = 12 2.96 1.69 1.14 0.84 0.89, W = 16 3.96 2.46 1.62 1.27 1.45.
static inline bool tsa_wide_slice_pays(int mode, int W, int nchains, int ncu) {
  if (W >= (mode == 0 ? 10 : 16)) return true;
  const int per_cu = mode == 0 ? (W - 2) / 2 : (W - 4) / 2;
  return nchains <= ncu * (per_cu < 1 ? 1 : per_cu);
}
