// tsa_team_rule.h -- how many waves sweep a chain in par order (k_team, or 1: k_sweep), and which kernel sweeps in pre-order
// with helper waves (k_team_pre, or k_sweep's helper form).  Plain C++, also compiled by the CPU tests.
#pragma once

// What the choice goes by.
struct TsaTeamRule {
  int asked;                // waves the caller asked for (0: automatic)
  int per_cu;               // chains per compute unit
  int units, units_float;   // wavefuls of lanes that one proposal per node takes, in tc mode and in the float modes
  int nint;
  bool moves;               // slice moves
  // chains that a compute unit's LDS holds: of a team's launch of sweeps and of its level loop, and of one wave each
  int lds, lds_loop, lds_one;
  int words;                // 64-bit words per label set
};
// Lanes of a proposal: two 64-bit words of its label sets a lane; the float modes always two lanes or more.
static constexpr int tsa_team_lanes(int W, int mode) { return W <= 2 ? (mode == 0 ? 1 : 2) : W / 2; }
// A launch of sweeps at one beta, a block of levels, the level loop.
enum TsaTeamKind { TSA_TEAM_SWEEPS, TSA_TEAM_BLOCK, TSA_TEAM_LOOP };

// Rounds of resident chains that per_cu chains take, at most `waves` and `lds` of them at once.
static inline int tsa_rounds(int per_cu, int waves, int lds) {
  const int most = waves < lds ? waves : lds;
  return (per_cu + most - 1) / (most > 0 ? most : 1);
}

// Sweeps with slice moves of five chains per unit and more (tc mode): two waves, or one where they take more rounds of
// resident chains.  The registers let 20 waves of k_team with slice moves share a unit with one word per label set and 16
// with more, of k_sweep 16 with one or two words, 12 with four, 4 with eight.  Ten sweeps and the energies, us, one wave /
// two, by chains per unit (*: a round more of teams):
//              6           7            8            10           12           16
//   sat40   271 / 199   270 / 200    272 / 204    311 / 232    317 / 332*   367 / 386*
//   sat60   324 / 227   327 / 228    328 / 235    379 / 265    385 / 370*   451 / 435*
//   sat70   386 / 275   388 / 276    389 / 282    452 / 444*   456 / 469*   534 / 592*
//   sat85   426 / 305   430 / 450*   432 / 483*   504 / 513*   510 / 570*   765 / 755*
//   sat100  468 / 493*  470 / 537*   473 / 554*   557 / 609*   563 / 774*   838 / 968*
//   sq10    263 / 189   265 / 190    267 / 197    315 / 298*   317 / 316*   466 / 381
// and of one sweep (12 chains per unit) sat60 64 / 70*, sat100 87 / 115*, sq10 59 / 69*.  With one word of several
// wavefuls and with four words a round more still pays from a few sweeps on.
static inline int tsa_team_moves_tc(const TsaTeamRule& r, int nsweeps) {
  if (r.nint < 64 && nsweeps < 2) return 1;
  const int team = r.words <= 1 ? 20 : 16, one = r.words <= 2 ? 16 : r.words <= 4 ? 12 : 4;
  if (tsa_rounds(r.per_cu, team / 2, r.lds) <= tsa_rounds(r.per_cu, one, r.lds_one)) return 2;
  if (r.words >= 4) return nsweeps < 2 ? 1 : 2;
  return r.words <= 1 && r.units >= 3 && nsweeps >= 4 ? 2 : 1;
}

// The lines lie where the measured times cross (par order, blocks of levels, 40 levels of one sweep, us):
//   chains  sat100: one wave / team of 2 / 4 / 8    sat60                     sq14 (8 words)
//      72            917 / 698 / 548 / 530          692 / 492 / 468 / 475      917 / 632 / 534 / 507
//    1024           1149 / 1097 / 901 / 1071        801 / 704 / 666 / 820     1298 / 1095 / 953 / 1085
//    2048           1491 / 1564 / 1338 / 1829       983 / 901 / 947 / 1329    1880 / 1694 / 1515 / 1872
//    4096           2413 / 2724 / 2416 / 3427      1482 / 1325 / 1603 / 2482  3425 / 3074 / 2799 / 3604
//    6144           3372 / 3908 / 3546 / 5093      1894 / 1891 / 2319 / 3620
// Eight waves pay while a compute unit has one chain; beyond that four where a tree's nodes (times the lanes of a
// proposal) fill them, else two; from 16 chains per unit on, one wave each hides its latency behind the others'.  With
// slice moves a chain holds a second cost cache, and from five chains per unit on two waves keep more of them resident
// (sat70, 2048 chains: 6.9 ms against 10.2 with four).
static inline int tsa_team_waves_tc(const TsaTeamRule& r, TsaTeamKind kind, int nsweeps) {
  if (r.per_cu > 16) return 1;
  const int big = r.units >= 5 && !r.moves ? 4 : 2;
  if (r.per_cu <= 1) return 8;
  if (r.per_cu <= 4) {
    // (a launch whose trees do not fill four waves: 1024 chains of reg60, one sweep: 36.9 us, two waves 31.4)
    if (kind == TSA_TEAM_SWEEPS && r.per_cu > 2 && r.units < 4) return 2;
    return 4;
  }
  // More chains than that per unit share it either way, and a team's launch starts with a pass over every chain for its
  // cost cache and stages the leaf sets per chain, so that it takes some sweeps before it is ahead.  Launch and
  // energies, us, one wave / team, at 8, 12 and 16 chains per unit:
  //   one sweep     sat30   36.9 / 40.3   41.8 / 48.2   45.8 / 62.0     sat100  56.0 / 66.7   64.3 / 80.0   87.5 / 98.4
  //   two           sat30   47.2 / 47.7   54.2 / 56.8   60.1 / 73.1     sat100  76.3 / 82.4   89.3 / 103.7  121.6 / 128.7
  //   four          sat30   67.1 / 62.5   78.1 / 75.4   87.6 / 102.8    sat100  115.5 / 119.9 135.6 / 152.4 190.5 / 192.3
  // And it takes more rounds where fewer teams than single waves are resident at once (28 waves of k_team a unit, 24 to 16
  // of k_sweep, and the LDS): then two waves per chain are never ahead (sat70, 12 per unit, eight sweeps 206 / 248), four
  // from eight sweeps on, and wide proposals (units >= 8) from two (sq14, 8 per unit, one sweep 87 / 97, two 110 / 111).
  const int waves_one = r.words <= 2 ? 24 : r.words <= 4 ? 20 : 16;
  const int rounds_one = tsa_rounds(r.per_cu, waves_one, r.lds_one);
  if (kind == TSA_TEAM_SWEEPS) {
    if (r.moves) return tsa_team_moves_tc(r, nsweeps);
    int least = r.units >= 8 || r.per_cu <= 6 ? 1 : r.per_cu <= 8 || r.words >= 4 ? 2 : 3;
    if (tsa_rounds(r.per_cu, 28 / big, r.lds) > rounds_one) {
      if (big == 2) return 1;
      if (r.units >= 8) least = rounds_one == 1 || r.per_cu > 12 ? 2 : 1;
      else least = r.per_cu <= 8 || rounds_one > 1 ? 8 : 16;
    }
    return nsweeps < least ? 1 : big;
  }
  // The loop's chains stay from its first level to its last, so all of them want to be resident at once: 16 waves of
  // k_team's loop a unit, 12 of k_sweep's (3072 chains of sat30, ten levels of ten sweeps: one wave 1324 us, two 1660;
  // 2048 chains of sat70, ten of five: 999 and 1296, 1792 chains 985 and 869).  With one sweep a level the loop's time is
  // the levels' folds, which a team makes beside the next sweep: a second round of it is worth it where the sweep is
  // short or wide (sq12, 2048 chains: one wave 635, four 560; sat30, 3072 chains: 674 and 626), unless the tree is
  // less than one scan of a wave.
  if (kind == TSA_TEAM_LOOP && !r.moves) {
    if (nsweeps < 2 && r.nint < 64) return 1;
    if (tsa_rounds(r.per_cu, 8, r.lds_loop) == 1) return 2;
    if (nsweeps < 2 && (r.words >= 4 || r.units < 4)) return big;
    if (tsa_rounds(r.per_cu, 12, r.lds_one) == 1 && !(r.units >= 8 && r.per_cu <= 6)) return 1;
  }
  return big;
}

// The float modes' visits are long enough for a team at any size, and their cost cache is the team's alone: four waves
// where a tree fills them, else two (gpu mode, four sweeps, one wave / two / four: 2048 chains of sat60 250 / 137 / 173,
// sat80 303 / 227 / 195; 8192 chains 628 / 414 / 513, 857 / 616 / 607).  The measured-time model's cost below its small
// rank is one addition, which a tree of a few dozen nodes hardly leaves: few sweeps there are over before a team's
// start has paid (17 nodes, 8192 chains, one sweep: 66 us against 99 with two waves and 149 with four).
static inline int tsa_team_waves_float(const TsaTeamRule& r, int mode, TsaTeamKind kind, int nsweeps) {
  if (r.per_cu <= 1) return 8;
  if (r.per_cu <= 4) return 4;
  if (mode == 2 && kind == TSA_TEAM_SWEEPS && r.nint < 48 && nsweeps < 4 && !r.moves) return 1;
  return r.moves || r.units_float < 9 ? 2 : 4;
}

// Waves per chain of a launch.  nsweeps: sweeps of the launch (TSA_TEAM_SWEEPS) or of a level.
static inline int tsa_team_waves(const TsaTeamRule& r, int mode, TsaTeamKind kind, int nsweeps) {
  if (r.asked > 0) return r.asked;
  return mode == 0 ? tsa_team_waves_tc(r, kind, nsweeps) : tsa_team_waves_float(r, mode, kind, nsweeps);
}

// Whether pre-order sweeps with helper waves run k_team_pre.  In tc mode and with a proposal on one lane its steps are no
// shorter than k_sweep's (a visit saves P's set and two look-ups and pushes entries of four words), only its start and its
// levels' ends, so that k_sweep is ahead from some sweeps on, the sooner the fewer chains there are.  k_sweep's time over
// k_team_pre's, launch of sweeps and energies / levels of the loop:
//                        4 sweeps    8     16     50     20 levels of 1    2     5     8 levels of 25
//   sat40,  16 chains      0.98    0.96   0.94   0.93          1.00      0.98  0.98       0.99
//           64             1.01    0.99   0.96   0.96          1.01      1.00  0.99       1.00
//          256             1.02    1.00   1.00   0.99          1.02      1.03  1.02       1.02
//   sat100, 16 (2 words)   1.01    1.00   0.98   0.97          1.00      1.00  0.99       1.01
//          256             1.02    1.01   1.00   0.99          1.07      1.04  1.03       1.02
// (43 chains of sat22, 65 levels of 50 sweeps: 32.3 ms with k_team_pre, 30.9 with k_sweep; 200 chains, 30 levels: 13.3,
// 13.5.)  W: 64-bit words per label set; sparse: fewer chains than half the compute units; nsweeps as above.
static inline bool tsa_pre_pays(int mode, int W, bool sparse, TsaTeamKind kind, int nsweeps) {
  if (mode != 0 || W > 2) return true;
  if (kind == TSA_TEAM_LOOP) return W > 1 || !sparse || nsweeps <= 2;
  return nsweeps <= (W > 1 || !sparse ? 8 : 4);
}
