// tsa_team.h -- par-order sweeps of small populations: one chain per workgroup, swept by a team of waves.
//
// k_sweep gives a chain one wave, which is right where thousands of chains hide each other's latency.  With a few
// chains per compute unit that wave's own chain of dependent steps is the time: a phase of the par sweep is a scan
// of every 64-node group one after the other, then visits of about 200 instructions and five dependent LDS round
// trips.  k_team spreads a chain over T = blockDim / 64 waves:
//   * scan: wave w takes the 64-node groups w, w + T, ... and appends their active nodes to the work list (an LDS
//     counter); workgroup barrier;
//   * visits: G lanes per proposal (two label words each, so a wide set costs a lane no more than a narrow one),
//     64 / G proposals per wave and round, counts summed inside a group by DPP quad permutes; workgroup barrier;
//   * random numbers: every node is visited once per sweep, so a sweep's Philox words are drawn before it by waves
//     that a phase of the previous sweep leaves without visits (rule bits and the 24-bit uniform in one word);
//   * node costs and sizes stay in LDS for the whole launch, rewritten by every accept: a visit counts only the
//     configuration after the move, an evaluation copies the cache, and in the float modes the two remaining node
//     costs of a visit are computed by two lanes at once (14 lse folds in a row become 4);
//   * slice moves: the current costs are the cache, the proposed ones one pass of the whole team, and one wave
//     folds both at once in its two halves (the reference's 32-lane order each).
// The phases, draws, floats and counters are those of the one-wave kernel (and of the CPU phase-by-phase sweep) bit
// for bit; visits of one phase touch disjoint words, so their order is free.
//
// Included by four translation units, one per SLICE and FULL variant.
#pragma once
#include "tsa_sweep.h"

// LDS byte offsets (same function on host and device): leaf sets ending where the record starts, the record, the work
// list, two buffers of draws, `caches` copies of the node-cost cache, then the node arrays.  A work-list entry is the
// node's children word, draw and cost word and its id (full: a visit then starts with the pivot's children word, two
// dependent LDS round trips earlier), or the id alone.
struct TsaTeamLds {
  int leaf, rec, wl, draw, cache, cache_bytes, nodes, bytes;
};
__host__ __device__ static inline TsaTeamLds tsa_team_lds(int m, int nint, int W, int chain_words, int mode,
                                                          int caches, int full) {
  const int nint4 = (nint + 3) & ~3, leafb = (m * W * 8 + 15) & ~15;
  TsaTeamLds L;
  L.leaf = leafb - m * W * 8;
  int b = leafb;
  L.rec = b;   b += chain_words * 8;
  L.wl = b;    b += nint4 * (full ? 16 : 2);
  L.draw = b;  b += 2 * nint4 * 4;
  L.cache = b;
  L.cache_bytes = nint4 * (mode == 0 ? 4 : 6);
  b += caches * L.cache_bytes;
  L.nodes = b; b += (2 * nint4 + TSA_PRI_PAD) * 2;  // priorities, parents
  L.bytes = (b + 15) & ~15;
  return L;
}
#define TSA_TEAM_STATIC_LDS 4096  // room for the static LDS of k_team and k_team_pre
// Copies of the cache a launch needs: the chain's, the proposed slice set's, and the level being folded.
static inline int tsa_team_caches(bool slice_moves, bool levels) { return 1 + (slice_moves ? 1 : 0) + (levels ? 1 : 0); }

// Node costs and masked sizes.  tc mode: both in one word (cost | size << 16; a tc cost is a count of labels);
// float modes: the cost's bits, and the sizes apart.
template <int MODE>
struct TsaTeamCache {
  uint32_t* a;
  uint16_t* z;
  __device__ __forceinline__ float cost(int i) const { return MODE == 0 ? (float)(a[i] & 0xFFFFu) : __uint_as_float(a[i]); }
  __device__ __forceinline__ int size(int i) const { return MODE == 0 ? (int)(a[i] >> 16) : (int)z[i]; }
  __device__ __forceinline__ void set(int i, float c, int s) const {
    if (MODE == 0) {
      a[i] = (uint32_t)c | ((uint32_t)s << 16);
    } else {
      a[i] = __float_as_uint(c);
      z[i] = (uint16_t)s;
    }
  }
};

// Lanes per proposal and label words per lane: two words a lane; the float modes always two lanes or more.
template <int W, int MODE>
struct TsaTeamShape {
  static constexpr int G = tsa_team_lanes(W, MODE);
  static constexpr int WL = W >= G ? W / G : 1;
};

template <int G>
__device__ __forceinline__ uint32_t tsa_group_sum(uint32_t x) {
  static_assert(G == 1 || G == 2 || G == 4, "groups inside a quad");
  if constexpr (G >= 2) x += tsa_lane_xor<1>(x);
  if constexpr (G >= 4) x += tsa_lane_xor<2>(x);
  return x;
}

// WL label words at p (16-byte aligned pairs).
struct alignas(16) TsaWords2 {
  uint64_t a, b;
};
template <int WL>
__device__ __forceinline__ void tsa_load_words(const uint64_t* p, uint64_t (&x)[WL]) {
  if constexpr (WL == 2) {
    const TsaWords2 v = *reinterpret_cast<const TsaWords2*>(p);
    x[0] = v.a;
    x[1] = v.b;
  } else {
    x[0] = p[0];
  }
}
template <int WL>
__device__ __forceinline__ void tsa_store_words(uint64_t* p, const uint64_t (&x)[WL]) {
  if constexpr (WL == 2) *reinterpret_cast<TsaWords2*>(p) = TsaWords2{x[0], x[1]};
  else p[0] = x[0];
}

// One sweep's draw of internal node v: the uniform's 24 bits above the rule's two.
__device__ __forceinline__ uint32_t tsa_team_draw(const TsaKParams& P, int v, uint32_t sw, uint32_t c) {
  const TsaU4 r = tsa_philox(TsaU4{(uint32_t)v, sw, c, 0u}, P.key0, P.key1);
  return (r.y & 0xFFFFFF00u) | (r.x >> 30);
}

// A visit's outcome: the children words of v and of the pivot after it, the pivot's cost word, the nodes it moved.
struct TsaTeamMove {
  uint32_t chv, chp, cp;
  int Pn, On, Mn;
  bool acc;
};
__device__ __forceinline__ bool tsa_team_has_rule(uint32_t chv, int m) {
  return (int)(chv & 0xFFFFu) >= m || (int)(chv >> 16) >= m;
}
// One proposal at the node of work-list entry w (children word, draw, cost word, id; it has a rule), by a group of G lanes
// (this one t): dE from the counts after the move and the cached costs before it, the Metropolis test, and when accepted
// the pivot's new set, the two children words and the cache (leader lane).  early(On, Mn): called once both are known,
// before the label sets arrive, for reads a caller wants in flight beside them.
template <int W, int MODE, bool SLICE, class Early>
__device__ __forceinline__ TsaTeamMove tsa_team_visit(const TsaKParams& P, uint64_t* lab, uint32_t* ch,
                                                      const TsaTeamCache<MODE>& cc, const uint64_t* S,
                                                      const float* s_lse, const float* s_ilse, const TsaMathTabs& T,
                                                      const uint4& w, float beta, int t, Early early) {
  constexpr int G = TsaTeamShape<W, MODE>::G, WL = TsaTeamShape<W, MODE>::WL, NC = MODE == 0 ? 4 : 10;
  const int m = P.m, vi = (int)w.w - m;
  const uint32_t chv = w.x, d = w.y;
  const int l = (int)(chv & 0xFFFFu), r = (int)(chv >> 16);
  const bool li = l >= m, ri = r >= m;
  const float costV = MODE == 0 ? (float)(w.z & 0xFFFFu) : __uint_as_float(w.z);
  const int b2 = (int)(d & 3u);
  const int rule = li && ri ? b2 : (li ? b2 >> 1 : 2 + (b2 >> 1));
  const int slotP = tsa_slot_p(rule), slotM = tsa_slot_m(rule);
  const int Pn = slotP ? r : l, On = slotP ? l : r, pi = Pn - m;
  const uint32_t chp = ch[pi], cp = cc.a[pi];
  const float costP = MODE == 0 ? (float)(cp & 0xFFFFu) : __uint_as_float(cp);
  const int szP = MODE == 0 ? (int)(cp >> 16) : (int)cc.z[pi];
  const int Mn = slotM ? (int)(chp >> 16) : (int)(chp & 0xFFFFu);
  const int Kn = slotM ? (int)(chp & 0xFFFFu) : (int)(chp >> 16);
  const int w0 = t * WL;
  const bool has = W >= G || t < W;  // (the float modes' second lane of a one-word set has none)
  uint64_t xd[WL], xo[WL], xk[WL], xm[WL], xx[WL];
  int pk[NC];
#pragma unroll
  for (int q = 0; q < NC; q++) pk[q] = 0;
  if (has) {
    tsa_load_words<WL>(lab + vi * W + w0, xd);
    tsa_load_words<WL>(lab + (On - m) * W + w0, xo);
    tsa_load_words<WL>(lab + (Kn - m) * W + w0, xk);
    tsa_load_words<WL>(lab + (Mn - m) * W + w0, xm);
  }
  early(On, Mn);
  if (has) {
#pragma unroll
    for (int i = 0; i < WL; i++) {
      xx[i] = tsa_xset(xk[i], xo[i], xm[i], xd[i]);
      uint64_t k = xk[i], o = xo[i], mm = xm[i], dd = xd[i], x = xx[i];
      if constexpr (SLICE) {
        const uint64_t nm = ~S[w0 + i];
        k &= nm;
        o &= nm;
        mm &= nm;
        dd &= nm;
        x &= nm;
      }
      pk[0] += tsa_popc64(dd);
      pk[1] += tsa_popc64(x);
      if constexpr (MODE == 0) {
        pk[2] += tsa_popc3<TSA_F_AB_NC>(k, o, x);
        pk[3] += tsa_popc3<TSA_F_AB_NC>(x, mm, dd);
      } else {
        tsa_count3(k, o, x, pk[2], pk[3], pk[4], pk[5]);
        tsa_count3(x, mm, dd, pk[6], pk[7], pk[8], pk[9]);
      }
    }
  }
  if constexpr (G > 1) {
#pragma unroll
    for (int q = 0; q < NC; q += 2) {
      const uint32_t z = tsa_group_sum<G>((uint32_t)pk[q] | ((uint32_t)pk[q + 1] << 16));
      pk[q] = (int)(z & 0xFFFFu);
      pk[q + 1] = (int)(z >> 16);
    }
  }
  const int sd = pk[0], sx = pk[1];
  float dE, newP, newV;
  if constexpr (MODE == 0) {
    dE = tsa_energy_tc_cached((int)costP, (int)costV, szP, sd, sx, pk[2], pk[3], P.model, s_lse);
    newP = (float)(sx + pk[2]);
    newV = (float)(sd + pk[3]);
  } else {
    // even lanes cost the new P = (K, O), odd lanes the new v = (P, M); then the even lanes fold the pair after the move
    // while the odd ones fold the pair before it
    const int q = t & 1;
    const float mine = tsa_node_cost_i<MODE>(q ? pk[6] : pk[2], q ? pk[7] : pk[3], q ? pk[8] : pk[4], q ? pk[9] : pk[5],
                                             P.model, T, s_ilse);
    const float other = tsa_lane_xor<1>(mine);
    newP = q ? other : mine;
    newV = q ? mine : other;
    const float h = tsa_lse_f(q ? costP : newP, q ? costV : newV, T);
    const float ho = tsa_lane_xor<1>(h);
    const float dtc = q ? ho - h : h - ho;
    const int sc0 = szP > sd ? szP : sd, sc1 = sx > sd ? sx : sd, scm = sc0 > sc1 ? sc0 : sc1;
    const float pw = ((float)scm > P.model.sc_target) ? P.model.sc_weight : 0.0f;
    dE = pw * (float)(sc1 - sc0) + dtc;
  }
  TsaTeamMove o{chv, chp, cp, Pn, On, Mn, tsa_metropolis(d, beta, dE, T.exp2)};
  if (o.acc) {
    if (has) tsa_store_words<WL>(lab + pi * W + w0, xx);
    o.chp = slotM ? ((chp & 0xFFFFu) | ((uint32_t)On << 16)) : ((chp & 0xFFFF0000u) | (uint32_t)On);
    o.chv = slotP ? ((chv & 0xFFFF0000u) | (uint32_t)Mn) : ((chv & 0xFFFFu) | ((uint32_t)Mn << 16));
    o.cp = MODE == 0 ? ((uint32_t)newP | ((uint32_t)sx << 16)) : __float_as_uint(newP);
    if (t == 0) {
      ch[pi] = o.chp;
      ch[vi] = o.chv;
      cc.set(pi, newP, sx);
      cc.set(vi, newV, sd);
    }
  }
  return o;
}

// 64-node groups of a wave's scan batch; rows of a pending level fold per phase (7 phases or so cover a tree of a few
// hundred nodes, so that the tracking wave's fold hides behind the phases of the next sweep).
#define TSA_TEAM_SCAN 2
#define TSA_TEAM_FOLD 2

// Slice moves by the whole team (tsa_slice_step's proposals and floats).  cc holds the costs and sizes of the tree
// under S, exact on entry and on return (cprop the spare copy; the two swap on an accepted move).  Every wave makes
// the proposal redundantly; the team evaluates the proposed slice set S2; wave 0 folds the current costs in lanes
// 0-31 and the proposed ones in lanes 32-63, so a proposal costs one pass of serial lse folds instead of two.
// Returns true when an evaluation was made; e (wave 0) is then the chain's as the step leaves it.  Every thread of the
// workgroup calls it, after a barrier; it ends with one.
template <int W, int MODE>
__device__ __forceinline__ bool tsa_team_slice_step(const TsaKParams& P, const uint64_t* lab, const uint32_t* ch,
                                                    uint64_t* S, uint64_t* S2, const uint64_t* lf,
                                                    const TsaMathTabs& T, float beta, uint32_t sw, uint32_t chain,
                                                    int tid, int NT, int* s_acc, TsaTeamCache<MODE>& cc,
                                                    TsaTeamCache<MODE>& cprop, int& nsp, int& nsa, TsaEvalOut& e) {
  const int lane = tid & 63, nint = P.nint;
  bool evaluated = false;
  for (int j = 0; j < P.slice_moves; j++) {
    // the current largest masked size, the nodes that have it, |S|
    int scm = 0, ncand = 0, ns = 0;
    for (int i = lane; i < nint; i += 64) {
      const int z = cc.size(i);
      ncand = z > scm ? 1 : ncand + (z == scm);
      scm = z > scm ? z : scm;
    }
    const int top = tsa_lane_max<64>(scm);
    ncand = tsa_lane_sum<64>(scm == top ? ncand : 0);
#pragma unroll
    for (int w = 0; w < W; w++) ns += __popcll(S[w]);
    const TsaU4 r1 = tsa_philox(TsaU4{0x10000u + 2u * (uint32_t)j, sw, chain, 0u}, P.key0, P.key1);
    const TsaU4 r2 = tsa_philox(TsaU4{0x10001u + 2u * (uint32_t)j, sw, chain, 0u}, P.key0, P.key1);
    int type;  // 0 add, 1 remove, 2 swap
    if (ns == 0) type = 0;
    else if (ns >= P.max_slices) type = (r1.x >> 31) ? 1 : 2;
    else type = r1.x < 0x80000000u ? 0 : (r1.x < 0xC0000000u ? 1 : 2);
    int ladd = -1, lrem = -1;
    if (type != 1 && ncand > 0 && top > 0) {
      // the (r1.y % ncand)-th internal node of maximal masked size, in node-id order
      int rr = (int)(r1.y % (uint32_t)ncand), node = -1;
      for (int b0 = 0; b0 < nint && node < 0; b0 += 64) {
        const int i = b0 + lane;
        const uint64_t b = __ballot(i < nint && cc.size(i) == top);
        const int n = __popcll(b);
        if (rr < n) node = b0 + tsa_nth_bit(b, rr);
        else rr -= n;
      }
      if (node >= 0) ladd = tsa_nth_label(lab + node * W, S, W, (int)(r1.z % (uint32_t)top));
    }
    if (type != 0) lrem = tsa_nth_label(S, nullptr, W, (int)(r1.w % (uint32_t)ns));
    if (type == 2 && ladd < 0) type = 1;
    if (type == 0 && ladd < 0) continue;  // uniform over the workgroup
    if (tid < W) {
      uint64_t x = S[tid];
      if (type != 1 && ladd >> 6 == tid) x |= 1ull << (ladd & 63);
      if (type != 0 && lrem >> 6 == tid) x &= ~(1ull << (lrem & 63));
      S2[tid] = x;
    }
    __syncthreads();
    for (int i = tid; i < nint; i += NT) {
      int Z;
      const float cst = tsa_node_eval<W, MODE>(P, lab, ch, S2, lf, T, i, Z);
      cprop.set(i, cst, Z);
    }
    __syncthreads();
    nsp++;
    if (tid < 64) {
      const bool hi = lane >= 32;
      const TsaTeamCache<MODE> f{hi ? cprop.a : cc.a, hi ? cprop.z : cc.z};
      const TsaEvalOut x =
          tsa_fold_finish(P, [&](int i) { return f.size(i); }, hi ? S2 : S, lf, W, T, lane & 31,
                          tsa_fold_rows([&](int i) { return f.cost(i); }, nint, T, lane & 31, -INFINITY, 0, (nint + 31) / 32));
      const float E = tsa_slice_energy(x, P);
      const auto from_lane = [](float y, int k) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(y), k)); };
      const bool acc = tsa_metropolis(r2.x, beta, from_lane(E, 32) - from_lane(E, 0), T.exp2);
      const int from = __builtin_amdgcn_readfirstlane(acc ? 32 : 0);
      e.lcost = from_lane(x.lcost, from);
      e.sc = __builtin_amdgcn_readlane(x.sc, from);
      e.ns = __builtin_amdgcn_readlane(x.ns, from);
      if (lane == 0) *s_acc = acc;
    }
    __syncthreads();
    evaluated = true;
    if (*s_acc) {
      nsa++;
      const TsaTeamCache<MODE> x = cc;
      cc = cprop;
      cprop = x;
      if (tid < W) S[tid] = S2[tid];
    }
    __syncthreads();
  }
  return evaluated;
}

// What the end of a level's fold reads, in LDS: tsa_team_fold_end is a call, and its frame would otherwise hold the
// kernel's whole parameter block.
struct TsaTeamFold {
  TsaLevels Lv;
  uint32_t* cost;      // the folded level's cache copy
  uint16_t* size;
  const uint64_t* S;   // its slice set (null: no slicing)
  const uint64_t* lf;
  TsaKParams P;
  TsaMathTabs T;
  int n, c;            // chains; this chain
};

// Rows from frow on of the pending fold, its end and the chain's arrival, by the tracking wave.  A call: inlined, the
// selection's registers (some 160) would be the sweeping loop's too.
template <int W, int MODE>
__device__ __attribute__((noinline)) TsaOwn tsa_team_fold_end(const TsaTeamFold* F, int frow, float facc, int ev,
                                                              int level, TsaOwn own, int slot) {
  const int lane = (int)threadIdx.x & 63;
  const TsaTeamCache<MODE> f{F->cost, F->size};
  const float acc = tsa_fold_rows([&](int i) { return f.cost(i); }, F->P.nint, F->T, lane & 31, facc, frow,
                                  (F->P.nint + 31) >> 5);
  const TsaEvalOut e = tsa_fold_finish(F->P, [&](int i) { return f.size(i); }, F->S, F->lf, W, F->T, lane & 31, acc);
  return tsa_level_arrive(F->Lv, F->n, F->c, ev, level, e.lcost, e.sc, e.ns, own, slot, lane);
}

template <int W, int MODE, bool SLICE, bool LVL, bool FULL>
__global__ void __launch_bounds__(512, MODE == 0 ? 4 : 2)
    k_team(TsaKParams P, uint64_t* __restrict__ rec, const uint64_t* __restrict__ leaf,
           const uint32_t* __restrict__ fix, int nchains, float beta1, uint32_t sweep0, int nsweeps,
           unsigned long long* __restrict__ stats, TsaEnergyOut eo, TsaLevels Lv) {
  extern __shared__ __align__(16) unsigned char tsa_tsm[];
  __shared__ float s_lse[64], s_ilse[TSA_ILSE];
  __shared__ uint64_t s_mt[TSA_MT_WORDS];
  __shared__ uint64_t s_S[8], s_S2[8];  // the slice set being folded; the proposed one
  __shared__ int s_cnt[2], s_draw, s_acc;
  __shared__ __align__(16) unsigned char s_fold[LVL ? sizeof(TsaTeamFold) : 16];
  static_assert(sizeof s_lse + sizeof s_ilse + sizeof s_mt + sizeof s_S + sizeof s_S2 + 16 + sizeof(TsaTeamFold) + 64 <=
                    TSA_TEAM_STATIC_LDS, "the plan leaves TSA_TEAM_STATIC_LDS bytes to the static arrays");
  constexpr int G = TsaTeamShape<W, MODE>::G, WL = TsaTeamShape<W, MODE>::WL;
  const int tid = threadIdx.x, NT = blockDim.x, T = NT >> 6, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = P.m, nint = P.nint, ngrp = (nint + 63) >> 6;
  const int c = P.chain0 + (int)blockIdx.x;  // (the grid is nchains - chain0 workgroups)
  const bool moves = SLICE && P.slice_moves > 0;
  const int ncache = 1 + (moves ? 1 : 0) + (LVL ? 1 : 0);
  const TsaTeamLds Lo = tsa_team_lds(m, nint, W, P.chain_words, MODE, ncache, FULL);
  uint64_t* const lf = reinterpret_cast<uint64_t*>(tsa_tsm + Lo.leaf);
  uint64_t* const base = reinterpret_cast<uint64_t*>(tsa_tsm + Lo.rec);
  uint64_t* const lab = base;
  uint32_t* const ch = reinterpret_cast<uint32_t*>(base + P.ch_off);
  uint64_t* const S = base + P.s_off;
  const uint64_t* const Sm = SLICE ? S : nullptr;
  uint32_t* const draws = reinterpret_cast<uint32_t*>(tsa_tsm + Lo.draw);
  const int nint4 = (nint + 3) & ~3;
  auto cache_at = [&](int k) {
    unsigned char* const p = tsa_tsm + Lo.cache + k * Lo.cache_bytes;
    return TsaTeamCache<MODE>{reinterpret_cast<uint32_t*>(p), reinterpret_cast<uint16_t*>(p + nint4 * 4)};
  };
  uint16_t* const pri = reinterpret_cast<uint16_t*>(tsa_tsm + Lo.nodes) + TSA_PRI_PAD;
  uint16_t* const par = pri + nint4;
  uint4* const wl4 = reinterpret_cast<uint4*>(tsa_tsm + Lo.wl);       // FULL
  uint16_t* const wl = reinterpret_cast<uint16_t*>(tsa_tsm + Lo.wl);  // else
  TsaTeamCache<MODE> cc = cache_at(0);
  TsaTeamCache<MODE> cprop = cache_at(moves ? 1 : 0);         // the proposed slice set's costs
  const TsaTeamCache<MODE> cfold = cache_at(ncache - 1);      // LVL: the level being folded
  const TsaMathTabs T_{s_mt, fix, fix + TSA_LOG2FIX_WORDS, s_mt + 32};

  // stage the tables, the leaf sets and the record
  uint64_t* const g = rec + (size_t)c * P.chain_words;
  if (tid < 64) s_lse[tid] = P.lse[tid];
  tsa_math_stage(s_mt);
  for (int i = tid; i < m * W; i += NT) lf[i] = leaf[i];
  {
    const uint4* const src = reinterpret_cast<const uint4*>(P.ganc ? P.gsrc + (size_t)P.ganc[c] * P.chain_words : g);
    uint4* const dst = reinterpret_cast<uint4*>(base);
    const int n16 = P.chain_words / 2;
    int i = tid;
    for (; i + 3 * NT < n16; i += 4 * NT) {  // four loads in flight per thread
      const uint4 a = src[i], b = src[i + NT], d = src[i + 2 * NT], e = src[i + 3 * NT];
      dst[i] = a;
      dst[i + NT] = b;
      dst[i + 2 * NT] = d;
      dst[i + 3 * NT] = e;
    }
    for (; i < n16; i += NT) dst[i] = src[i];
  }
  if (tid == 0) {
    s_cnt[0] = s_cnt[1] = 0;
    s_draw = 0;
  }
  // the level loop, a block of levels (eo.blk), or the launch's one level
  const bool blocked = !LVL && eo.blk.n > 0;
  const int nsw = LVL ? Lv.total : (blocked ? eo.blk.total : nsweeps);
  int lv = 0, left = LVL ? Lv.niters[0] : (blocked ? eo.blk.niters[0] : nsweeps);
  float beta = LVL ? Lv.beta[0] : (blocked ? eo.blk.beta[0] : beta1);
  for (int i = tid; i < nint; i += NT) draws[i] = tsa_team_draw(P, m + i, sweep0, (uint32_t)c);
  __syncthreads();
  if constexpr (MODE != 0) tsa_ilse_stage(s_ilse, T_);
  for (int i = tid; i < nint; i += NT) {
    const uint32_t cw = ch[i];
    const int l = (int)(cw & 0xFFFFu), r = (int)(cw >> 16);
    if (l >= m) par[l - m] = (uint16_t)(m + i);
    if (r >= m) par[r - m] = (uint16_t)(m + i);
    int Z;
    const float cst = tsa_node_eval<W, MODE>(P, lab, ch, Sm, lf, T_, i, Z);
    cc.set(i, cst, Z);
  }
  if (tid == 0) {
    par[nint - 1] = 0u;  // (leaf id 0: no parent, see tsa_pri_key)
    pri[-1] = 0;
  }

  // the level loop: the last wave tracks the chain; its fold of an evaluated level runs a few rows per phase of
  // the sweeps that follow (frow: the next row, -1 none)
  const bool tracker = LVL && wv == T - 1;
  const int rows = (nint + 31) >> 5;
  int frow = -1, fev = 0, flev = 0, fslot = 0;
  float facc = -INFINITY;
  TsaOwn own{INFINITY, -1};
  if (tracker && !Lv.reset) own = TsaOwn{Lv.own[c], Lv.bslot[c]};
  if (tracker && Lv.tinit && c == 0) {
    // the session's start: its stores precede this chain's first arrival (release), which every trace row's
    // writer waits for (acquire)
    unsigned long long* const tr = reinterpret_cast<unsigned long long*>(Lv.trace);
    for (int i = lane; i < Lv.trace_words; i += 64) tr[i] = 0ull;
    for (int i = lane; i < Lv.best_words; i += 64) Lv.best[i] = 0ull;
    if (lane == 0) {
      Lv.tinit->best_score = INFINITY;
      Lv.tinit->best_chain = -1;
      Lv.tinit->best_level = -1;
      Lv.tinit->snap = -1;
      *Lv.ticks0 = wall_clock64();
    }
  }
  TsaTeamFold* const F = reinterpret_cast<TsaTeamFold*>(s_fold);
  if constexpr (LVL) {
    if (tid == 0) *F = TsaTeamFold{Lv, cfold.a, cfold.z, SLICE ? s_S : nullptr, lf, P, T_, nchains, c};
  }
  auto fold_end = [&]() {
    own = tsa_team_fold_end<W, MODE>(F, frow, facc, fev, flev, own, fslot);
    frow = -1;
  };

  int np = 0, na = 0, nst = 0, nv = 0, nsp = 0, nsa = 0;
  int ph = 0;
  TsaEvalOut last_e{};
  bool have_e = false;
  const int t = lane & (G - 1), gsub = lane / G;
  constexpr int GPW = 64 / G;  // proposals per wave and round
  for (int s = 0; s < nsw; s++) {
    const uint32_t sw = sweep0 + (uint32_t)s;
    const uint32_t hs = tsa_sweep_hash(sw, (uint32_t)c, P.key0);
    for (int i = tid; i < nint; i += NT) pri[i] = (uint16_t)tsa_par_pri((uint32_t)(m + i), hs);
    __syncthreads();
    if (tid == 0) s_draw = 0;  // (this sweep's draws are complete; the next ones start after the next barrier)
    const uint32_t* const dr = draws + (s & 1) * nint4;
    uint32_t* const dn = draws + ((s + 1) & 1) * nint4;
    const bool draw_next = s + 1 < nsw;
    auto draw_some = [&]() -> bool {  // 64 of the next sweep's draws; false when none is left
      int k = 0;
      if (lane == 0) k = atomicAdd(&s_draw, 1);
      k = __builtin_amdgcn_readfirstlane(k);
      if (k >= ngrp) return false;
      const int i = k * 64 + lane;
      if (i < nint) dn[i] = tsa_team_draw(P, m + i, sw + 1u, (uint32_t)c);
      return true;
    };
    bool draws_left = draw_next;
    int unvisited = nint;
    const uint32_t m1 = (uint32_t)m - 1u;
    while (unvisited > 0) {
      // scan: this wave's groups, TSA_TEAM_SCAN at a time (every read of a batch in flight at once)
      for (int g0 = wv; g0 < ngrp; g0 += T * TSA_TEAM_SCAN) {
        uint32_t pv[TSA_TEAM_SCAN], pw[TSA_TEAM_SCAN], kp[TSA_TEAM_SCAN], kl[TSA_TEAM_SCAN], kr[TSA_TEAM_SCAN];
        uint4 en[TSA_TEAM_SCAN];
#pragma unroll
        for (int q = 0; q < TSA_TEAM_SCAN; q++) {
          const int gi = g0 + q * T;
          pv[q] = pw[q] = 0u;
          en[q] = uint4{0u, 0u, 0u, 0u};
          if (gi < ngrp) {  // uniform
            const int i = gi * 64 + lane, ic = i < nint ? i : nint - 1;
            pv[q] = pri[ic];
            pw[q] = par[ic];
            en[q] = uint4{ch[ic], 0u, 0u, (uint32_t)(m + ic)};
            if constexpr (FULL) {
              en[q].y = dr[ic];
              en[q].z = cc.a[ic];
            }
          }
        }
#pragma unroll
        for (int q = 0; q < TSA_TEAM_SCAN; q++) {
          kp[q] = kl[q] = kr[q] = 0u;
          if (g0 + q * T < ngrp) {
            kp[q] = tsa_pri_key(pri, m1, pw[q]);
            kl[q] = tsa_pri_key(pri, m1, en[q].x & 0xFFFFu);
            kr[q] = tsa_pri_key(pri, m1, en[q].x >> 16);
          }
        }
        uint64_t bb[TSA_TEAM_SCAN];
        int tot = 0;
#pragma unroll
        for (int q = 0; q < TSA_TEAM_SCAN; q++) {
          const int here = nint - (g0 + q * T) * 64;  // nodes from this group on
          const uint64_t vm = here >= 64 ? ~0ull : here > 0 ? (1ull << here) - 1ull : 0ull;
          bb[q] = __ballot(tsa_scan_active(en[q].w, pv[q], kp[q], kl[q], kr[q])) & vm;
          tot += __popcll(bb[q]);
        }
        if (tot == 0) continue;
        int at = 0;
        if (lane == 0) at = atomicAdd(&s_cnt[ph & 1], tot);
        at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
        for (int q = 0; q < TSA_TEAM_SCAN; q++) {
          if ((bb[q] >> lane) & 1ull) {
            if constexpr (FULL) wl4[at + tsa_rank(bb[q])] = en[q];
            else wl[at + tsa_rank(bb[q])] = (uint16_t)en[q].w;
          }
          at += __popcll(bb[q]);
        }
      }
      __syncthreads();
      const int j0 = wv * GPW;
      uint4 w{};
      if constexpr (FULL) w = wl4[j0 + gsub < nint4 ? j0 + gsub : 0];  // (beside the count; used when there is such an entry)
      const int cnt = s_cnt[ph & 1];
      if (cnt == 0) break;  // (uniform; only a record that holds no tree)
      if (tid == 0) s_cnt[(ph + 1) & 1] = 0;  // (last read before the previous phase's second barrier)
      nst++;
      unvisited -= cnt;
      ph++;
      if (LVL && tracker && frow >= 0) {
        if (frow < rows) {
          const int r1 = frow + TSA_TEAM_FOLD < rows ? frow + TSA_TEAM_FOLD : rows;
          facc = tsa_fold_rows([&](int i) { return cfold.cost(i); }, nint, T_, lane & 31, facc, frow, r1);
          frow = r1;
        } else {
          fold_end();
        }
      }
      if (j0 >= cnt && draws_left) draws_left = draw_some();
      for (int j1 = j0; j1 < cnt; j1 += T * GPW) {
        const int j = j1 + gsub;
        if (j >= cnt) continue;  // whole groups
        if constexpr (!FULL) {
          w.w = wl[j];
          const int i = (int)w.w - m;
          w.x = ch[i];
          w.y = dr[i];
          w.z = cc.a[i];
        } else if (j1 > j0) {
          w = wl4[j];
        }
        const int v = (int)w.w, vi = v - m;
        if (tsa_team_has_rule(w.x, m)) {
          const TsaTeamMove o = tsa_team_visit<W, MODE, SLICE>(P, lab, ch, cc, S, s_lse, s_ilse, T_, w, beta, t, [](int, int) {});
          if (t == 0) {
            np++;
            na += o.acc;
            if (o.acc && o.On >= m) par[o.On - m] = (uint16_t)o.Pn;
            if (o.acc && o.Mn >= m) par[o.Mn - m] = (uint16_t)v;
          }
        }
        if (t == 0) {
          nv++;
          pri[vi] = 0;
        }
      }
      __syncthreads();
    }
    if constexpr (SLICE) {
      have_e = false;
      if (moves && (sw + 1u) % (uint32_t)P.slice_every == 0u) {
        have_e = tsa_team_slice_step<W, MODE>(P, lab, ch, S, s_S2, lf, T_, beta, sw, (uint32_t)c, tid, NT, &s_acc, cc,
                                              cprop, nsp, nsa, last_e);
      }
    }
    while (draws_left && draw_some()) {
    }
    if constexpr (LVL) {
      if (--left == 0) {  // the level's last sweep
        const int ev = F->Lv.eval[lv];
        if (ev >= 0) {
          if (tracker && frow >= 0) fold_end();  // the previous level's, not yet done
          __syncthreads();
          for (int i = tid; i < nint; i += NT) {
            cfold.a[i] = cc.a[i];
            if (MODE != 0) cfold.z[i] = cc.z[i];
          }
          if (SLICE && tid < W) s_S[tid] = S[tid];
          if (tracker) {
            fslot = own.slot < 0 ? 0 : own.slot ^ 1;
            tsa_level_keep(F->Lv, P, base, nchains, c, fslot, lane, 64);
            frow = 0;
            facc = -INFINITY;
            fev = ev;
            flev = lv;
          }
        }
        if (++lv < F->Lv.nlev) {
          beta = F->Lv.beta[lv];
          left = F->Lv.niters[lv];
        }
      }
    } else {
      if (blocked && --left == 0) {  // a block's level ends: its snapshot (node costs, sizes, children words)
        if (eo.blk.cost[lv]) {
          float* const gc = eo.blk.cost[lv] + (size_t)c * nint4;
          uint16_t* const gz = eo.blk.z[lv] + (size_t)c * nint4;
          uint32_t* const gch = eo.blk.ch[lv] + (size_t)c * nint;
          for (int i = tid; i < nint; i += NT) {
            gc[i] = cc.cost(i);
            gz[i] = (uint16_t)cc.size(i);
            gch[i] = ch[i];
          }
        }
        if (++lv < eo.blk.n) {
          beta = eo.blk.beta[lv];
          left = eo.blk.niters[lv];
        }
      }
    }
  }
  __syncthreads();
  if constexpr (LVL) {
    if (tracker) {
      if (frow >= 0) fold_end();
      if (lane == 0) {
        F->Lv.own[c] = own.s;
        F->Lv.bslot[c] = own.slot;
      }
    }
  }
  // what the launch leaves of the chain's energies: node costs for the fold kernel, or the fold by wave 0
  if (eo.cost) {
    float* const gc = eo.cost + (size_t)c * nint4;
    uint16_t* const gz = eo.z + (size_t)c * nint4;
    for (int i = tid; i < nint; i += NT) {
      gc[i] = cc.cost(i);
      gz[i] = (uint16_t)cc.size(i);
    }
  } else if (eo.lc && wv == 0) {
    const TsaEvalOut e =
        have_e ? last_e
               : tsa_fold_finish(P, [&](int i) { return cc.size(i); }, Sm, lf, W, T_, lane & 31,
                                 tsa_fold_rows([&](int i) { return cc.cost(i); }, nint, T_, lane & 31, -INFINITY, 0, rows));
    if (lane == 0) {
      eo.lc[c] = e.lcost;
      eo.sc[c] = e.sc;
      eo.ns[c] = e.ns;
    }
  }
  if (eo.ch) {
    uint32_t* const gch = eo.ch + (size_t)c * nint;
    for (int i = tid; i < nint; i += NT) gch[i] = ch[i];
  }
  for (int i = tid; i < P.chain_words / 2; i += NT)
    reinterpret_cast<uint4*>(g)[i] = reinterpret_cast<const uint4*>(base)[i];
  const long long sp_ = tsa_wave_sum(np), sa_ = tsa_wave_sum(na), sv_ = tsa_wave_sum(nv);
  if (lane == 0) {  // counters spread over TSA_STAT_SLOTS addresses each, summed by the host
    unsigned long long* st = stats + ((c * 8 + wv) & (TSA_STAT_SLOTS - 1));
    atomicAdd(&st[TSA_ST_PROP * TSA_STAT_SLOTS], (unsigned long long)sp_);
    atomicAdd(&st[TSA_ST_ACC * TSA_STAT_SLOTS], (unsigned long long)sa_);
    atomicAdd(&st[TSA_ST_VISITS * TSA_STAT_SLOTS], (unsigned long long)sv_);
    atomicAdd(&st[TSA_ST_BUSY * TSA_STAT_SLOTS], (unsigned long long)sv_);
    if (wv == 0) {
      atomicAdd(&st[TSA_ST_STEPS * TSA_STAT_SLOTS], (unsigned long long)nst);
      if (SLICE) {
        atomicAdd(&st[TSA_ST_SPROP * TSA_STAT_SLOTS], (unsigned long long)nsp);
        atomicAdd(&st[TSA_ST_SACC * TSA_STAT_SLOTS], (unsigned long long)nsa);
      }
    }
  }
}

template <int W, int MODE, bool SLICE, bool LVL, bool FULL>
static hipError_t launch_team_t(const TsaLaunch& L, const TsaKParams& P, uint64_t* rec, const uint64_t* leaf,
                                const uint32_t* fix, int nchains, float beta, uint32_t sweep0, int nsweeps,
                                unsigned long long* stats, const TsaEnergyOut& eo, hipStream_t st, hipEvent_t e0,
                                hipEvent_t e1, const TsaLevels* lv, int* res) {
  const int caches = tsa_team_caches(SLICE && P.slice_moves > 0, LVL);
  const size_t smem = (size_t)tsa_team_lds(P.m, P.nint, W, P.chain_words, MODE, caches, FULL).bytes;
  const int threads = 64 * L.team;
  const void* const fn = reinterpret_cast<const void*>(&k_team<W, MODE, SLICE, LVL, FULL>);
  if (smem > 65536) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
  }
  if (res) return hipOccupancyMaxActiveBlocksPerMultiprocessor(res, fn, threads, smem);  // a query, no launch
  if (P.chain0 < 0 || P.chain0 >= nchains) return hipErrorInvalidValue;
  if (eo.blk.n > 0 && (LVL || eo.blk.n > TSA_BLOCK_MAX || eo.blk.total != nsweeps)) return hipErrorInvalidValue;
  hipExtLaunchKernelGGL((k_team<W, MODE, SLICE, LVL, FULL>), dim3(nchains - P.chain0), dim3(threads), (uint32_t)smem, st, e0,
                        e1, 0u, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, lv ? *lv : TsaLevels{});
  return hipGetLastError();
}

template <int W, bool SLICE, bool FULL>
static hipError_t launch_team_w(const TsaLaunch& L, int mode, const TsaKParams& P, uint64_t* rec, const uint64_t* leaf,
                                const uint32_t* fix, int nchains, float beta, uint32_t sweep0, int nsweeps,
                                unsigned long long* stats, const TsaEnergyOut& eo, hipStream_t st, hipEvent_t e0,
                                hipEvent_t e1, const TsaLevels* lv, int* res) {
#define TSA_TEAM_GO(MODE)                                                                                              \
  return lv ? launch_team_t<W, MODE, SLICE, true, FULL>(L, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats,   \
                                                        eo, st, e0, e1, lv, res)                                       \
            : launch_team_t<W, MODE, SLICE, false, FULL>(L, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats,  \
                                                         eo, st, e0, e1, lv, res)
  if (mode == 0) TSA_TEAM_GO(0);
  if (mode == 1) TSA_TEAM_GO(1);
  TSA_TEAM_GO(2);
#undef TSA_TEAM_GO
}

template <bool SLICE, bool FULL>
static hipError_t tsa_launch_team_t(const TsaLaunch& L, int mode, const TsaKParams& P, uint64_t* rec,
                                    const uint64_t* leaf, const uint32_t* fix, int nchains, float beta,
                                    uint32_t sweep0, int nsweeps, unsigned long long* stats, const TsaEnergyOut& eo,
                                    hipStream_t st, hipEvent_t e0, hipEvent_t e1, const TsaLevels* lv, int* res) {
  switch (L.W) {
    case 1: return launch_team_w<1, SLICE, FULL>(L, mode, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1, lv, res);
    case 2: return launch_team_w<2, SLICE, FULL>(L, mode, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1, lv, res);
    case 4: return launch_team_w<4, SLICE, FULL>(L, mode, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1, lv, res);
    case 8: return launch_team_w<8, SLICE, FULL>(L, mode, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1, lv, res);
    default: return hipErrorInvalidValue;
  }
}
