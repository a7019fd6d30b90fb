// tsa_team_rule.h -- how many waves sweep a chain in par order (k_team, or 1: k_sweep).  Plain C++, also compiled by the
// CPU tests.
#pragma once

// What the choice goes by.
struct TsaTeamRule {
  int asked;                // waves the caller asked for (0: automatic)
  int per_cu;               // chains per compute unit
  int units, units_float;   // wavefuls of lanes that one proposal per node takes, in tc mode and in the float modes
  int nint;
  bool moves;               // slice moves
};
// Lanes of a proposal: two 64-bit words of its label sets a lane; the float modes always two lanes or more.
static constexpr int tsa_team_lanes(int W, int mode) { return W <= 2 ? (mode == 0 ? 1 : 2) : W / 2; }
// A launch of sweeps at one beta, a block of levels, the level loop.
enum TsaTeamKind { TSA_TEAM_SWEEPS, TSA_TEAM_BLOCK, TSA_TEAM_LOOP };

// The lines lie where the measured times cross (par order, blocks of levels, 40 levels of one sweep, us):
//   chains  sat100: one wave / team of 2 / 4 / 8    sat60                     sq14 (8 words)
//      72            917 / 698 / 548 / 530          692 / 492 / 468 / 475      917 / 632 / 534 / 507
//    1024           1149 / 1097 / 901 / 1071        801 / 704 / 666 / 820     1298 / 1095 / 953 / 1085
//    2048           1491 / 1564 / 1338 / 1829       983 / 901 / 947 / 1329    1880 / 1694 / 1515 / 1872
//    4096           2413 / 2724 / 2416 / 3427      1482 / 1325 / 1603 / 2482  3425 / 3074 / 2799 / 3604
//    6144           3372 / 3908 / 3546 / 5093      1894 / 1891 / 2319 / 3620
// Eight waves pay while a compute unit has one chain; beyond that four where a tree's nodes (times the lanes of a
// proposal) fill them, else two; from 16 chains per unit on, one wave each hides its latency behind the others'.  With
// slice moves a chain holds a second cost cache, and from five chains per unit on two waves keep all of them resident
// (sat70, 2048 chains: 6.9 ms against 10.2 with four).
static inline int tsa_team_waves_tc(const TsaTeamRule& r, TsaTeamKind kind, int nsweeps) {
  if (r.per_cu > 16) return 1;
  const int big = r.units >= 5 && !r.moves ? 4 : 2;
  if (r.per_cu <= 1) return 8;
  if (r.per_cu <= 4) {
    // (a launch whose trees do not fill four waves: 1024 chains of reg60, one sweep: 36.9 us, two waves 31.4)
    if (kind == TSA_TEAM_SWEEPS && r.per_cu > 2 && r.units < 5) return 2;
    return 4;
  }
  // More chains than that per unit share it either way, and a team's launch starts with a pass over every chain for its
  // cost cache and stages the leaf sets per chain, so that it takes some sweeps before it is ahead.  Launch and
  // energies, us, one wave / team, at 8, 12 and 16 chains per unit:
  //   one sweep     sat30   36.9 / 40.3   41.8 / 48.2   45.8 / 62.0     sat100  56.0 / 66.7   64.3 / 80.0   87.5 / 98.4
  //   two           sat30   47.2 / 47.7   54.2 / 56.8   60.1 / 73.1     sat100  76.3 / 82.4   89.3 / 103.7  121.6 / 128.7
  //   four          sat30   67.1 / 62.5   78.1 / 75.4   87.6 / 102.8    sat100  115.5 / 119.9 135.6 / 152.4 190.5 / 192.3
  // Wide proposals (units >= 8) are ahead from the first (reg250: 92 / 70, 137 / 105, 170 / 123).
  if (kind == TSA_TEAM_SWEEPS) {
    if (r.moves) return r.nint < 64 && nsweeps < 2 ? 1 : big;
    if (r.units >= 8 || r.per_cu <= 6) return big;
    const int least = r.per_cu <= 8 ? 2 : r.per_cu <= 12 ? (r.units >= 5 ? 16 : 3) : (r.units >= 5 ? 8 : 16);
    return nsweeps < least ? 1 : big;
  }
  // The loop's chains stay from its first level to its last: one wave keeps twelve of them resident on a unit, two
  // waves eight (sat30, 3072 chains, ten levels of ten sweeps: 1324 against 1660 us), four waves four (sat100: 2646
  // against 3656).
  if (kind == TSA_TEAM_LOOP && !r.moves && r.units < 8) {
    if (r.per_cu > (r.units >= 5 ? 6 : 8)) return 1;
    if (r.nint < 64 && nsweeps < 2) return 1;
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
