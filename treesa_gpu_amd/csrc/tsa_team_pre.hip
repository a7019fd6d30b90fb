// tsa_team_pre.hip -- pre-order sweeps of chains in LDS by one sweeping wave and helpers (k_team_pre), without slicing.
//
// A pre-order sweep is a chain of dependent steps (a node is visited after its parent; 20 to 30 steps for trees of a few
// hundred nodes), so its time is the latency of a step.  Wave 0 sweeps; three helper waves draw the next sweep's random
// numbers beside it and, in the level loop, fold and select an evaluated level.  Against the one-wave kernel's
// helper form a step is shorter by
//   * visits of k_team's kind: lane groups of two words each, the costs before the move from the cache in every mode (a
//     float-mode visit's four node costs become two, on two lanes at once);
//   * work-list entries that carry the node's children word, draw and cost word: a visit knows its children's (the
//     pivot's are in hand, the other child's and the moved grandchild's are read beside the label sets), so that a
//     step starts with the pivot's children word instead of three dependent look-ups.
// Steps, draws, floats and counters are those of the one-wave kernel (up to 64 ready nodes from the top of the list a
// step, children pushed in its order).
#include "tsa_team.h"

// LDS byte offsets: as tsa_team_lds, with room for a frontier (at most half the nodes: none is another's ancestor).
struct TsaTeamPreLds {
  int leaf, rec, wl, draw, cache, cache_bytes, bytes;
};
__host__ __device__ static inline TsaTeamPreLds tsa_team_pre_lds(int m, int nint, int W, int chain_words, int mode,
                                                                 int caches) {
  const int nint4 = (nint + 3) & ~3, leafb = (m * W * 8 + 15) & ~15;
  TsaTeamPreLds L;
  L.leaf = leafb - m * W * 8;
  int b = leafb;
  L.rec = b;   b += chain_words * 8;
  L.wl = b;    b += (nint4 / 2 + 4) * 16;
  L.draw = b;  b += 2 * nint4 * 4;
  L.cache = b;
  L.cache_bytes = nint4 * (mode == 0 ? 4 : 6);
  b += caches * L.cache_bytes;
  L.bytes = (b + 15) & ~15;
  return L;
}

template <int W, int MODE, bool LVL>
__global__ void __launch_bounds__(64 * (1 + TSA_DRAW_HELPERS))
    k_team_pre(TsaKParams P, uint64_t* __restrict__ rec, const uint64_t* __restrict__ leaf,
               const uint32_t* __restrict__ fix, int nchains, float beta1, uint32_t sweep0, int nsweeps,
               unsigned long long* __restrict__ stats, TsaEnergyOut eo, TsaLevels Lv) {
  extern __shared__ __align__(16) unsigned char tsa_tsm[];
  __shared__ float s_lse[64], s_ilse[TSA_ILSE];
  __shared__ uint64_t s_mt[TSA_MT_WORDS];
  __shared__ __align__(16) unsigned char s_fold[LVL ? sizeof(TsaTeamFold) : 16];
  static_assert(sizeof s_lse + sizeof s_ilse + sizeof s_mt + sizeof(TsaTeamFold) + 64 <= TSA_TEAM_STATIC_LDS,
                "the plan leaves TSA_TEAM_STATIC_LDS bytes to the static arrays");
  constexpr int G = TsaTeamShape<W, MODE>::G, GPW = 64 / G, R = G;  // R rounds of GPW proposals hold a step's 64
  const int tid = threadIdx.x, NT = blockDim.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = P.m, nint = P.nint, nint4 = (nint + 3) & ~3;
  const int c = P.chain0 + (int)blockIdx.x;  // (the grid is nchains - chain0 workgroups)
  const TsaTeamPreLds Lo = tsa_team_pre_lds(m, nint, W, P.chain_words, MODE, 1 + (LVL ? 1 : 0));
  uint64_t* const lf = reinterpret_cast<uint64_t*>(tsa_tsm + Lo.leaf);
  uint64_t* const base = reinterpret_cast<uint64_t*>(tsa_tsm + Lo.rec);
  uint64_t* const lab = base;
  uint32_t* const ch = reinterpret_cast<uint32_t*>(base + P.ch_off);
  uint4* const wl = reinterpret_cast<uint4*>(tsa_tsm + Lo.wl);
  uint32_t* const draws = reinterpret_cast<uint32_t*>(tsa_tsm + Lo.draw);
  auto cache_at = [&](int k) {
    unsigned char* const p = tsa_tsm + Lo.cache + k * Lo.cache_bytes;
    return TsaTeamCache<MODE>{reinterpret_cast<uint32_t*>(p), reinterpret_cast<uint16_t*>(p + nint4 * 4)};
  };
  const TsaTeamCache<MODE> cc = cache_at(0), cfold = cache_at(LVL ? 1 : 0);
  const TsaMathTabs T_{s_mt, fix, fix + TSA_LOG2FIX_WORDS, s_mt + 32};
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
  const int nsw = LVL ? Lv.total : nsweeps;
  int lv = 0, left = LVL ? Lv.niters[0] : nsweeps;
  float beta = LVL ? Lv.beta[0] : beta1;
  for (int i = tid; i < nint; i += NT) draws[i] = tsa_team_draw(P, m + i, sweep0, (uint32_t)c);
  __syncthreads();
  if constexpr (MODE != 0) tsa_ilse_stage(s_ilse, T_);
  for (int i = tid; i < nint; i += NT) {
    int Z;
    const float cst = tsa_node_eval<W, MODE>(P, lab, ch, nullptr, lf, T_, i, Z);
    cc.set(i, cst, Z);
  }
  const bool tracker = LVL && wv == 1;
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
    if (tid == 0) *F = TsaTeamFold{Lv, cfold.a, cfold.z, nullptr, lf, P, T_, nchains, c};
  }
  __syncthreads();
  auto keep_costs = [&]() {  // an evaluated level's costs, which wave 1 folds beside the next sweep
    for (int i = tid; i < nint; i += NT) {
      cfold.a[i] = cc.a[i];
      if (MODE != 0) cfold.z[i] = cc.z[i];
    }
  };
  // The level's entry of the schedule, and the next one's, read a level ahead: at a level's end every wave goes by it at
  // once, where a read would be two round trips to memory on the sweeping wave's path (256 chains of sat100, 100 levels of
  // one sweep, 2147 -> 2081 us).
  int ev = 0, ev_next = 0, left_next = 0;
  float beta_next = beta;
  auto read_ahead = [&]() {
    const int k = lv + 1 < Lv.nlev ? lv + 1 : lv;
    ev_next = Lv.eval[k];
    left_next = Lv.niters[k];
    beta_next = Lv.beta[k];
  };
  auto next_level = [&]() {
    lv++;
    ev = ev_next;
    left = left_next;
    beta = beta_next;
    read_ahead();
  };
  if constexpr (LVL) {
    ev = Lv.eval[0];
    read_ahead();
  }
  int np = 0, na = 0, nst = 0, nv = 0;
  // The sweeping wave and the helpers run loops of their own, which meet at the same workgroup barriers: one per sweep,
  // one more at an evaluated level's end.
  if (wv > 0) {
    for (int s = 0; s < nsw; s++) {
      if (s + 1 < nsw) {
        uint32_t* const dn = draws + ((s + 1) & 1) * nint4;
        for (int i = tid - 64; i < nint; i += NT - 64) dn[i] = tsa_team_draw(P, m + i, sweep0 + (uint32_t)s + 1u, (uint32_t)c);
      }
      __syncthreads();
      if constexpr (LVL) {
        if (--left == 0) {  // the level's last sweep
          if (ev >= 0) {
            keep_costs();
            const int slot = own.slot < 0 ? 0 : own.slot ^ 1;
            if (wv == 1) tsa_level_keep(F->Lv, P, base, nchains, c, slot, lane, 64);
            __syncthreads();
            if (wv == 1) own = tsa_team_fold_end<W, MODE>(F, 0, -INFINITY, ev, lv, own, slot);
          }
          next_level();
        }
      }
    }
  } else {
    const int t = lane & (G - 1), gsub = lane / G;
    for (int s = 0; s < nsw; s++) {
      const uint32_t* const dr = draws + (s & 1) * nint4;
      if (lane == 0) wl[0] = uint4{ch[nint - 1], dr[nint - 1], cc.a[nint - 1], (uint32_t)(2 * m - 2)};
      int sp = 1;
      tsa_wave_sync();
      while (sp > 0) {
        const int k = sp < 64 ? sp : 64, b0 = sp - k;
        uint4 e[R];
#pragma unroll
        for (int q = 0; q < R; q++)  // every entry of the step is read before a push overwrites it
          if (q * GPW < k) e[q] = wl[b0 + q * GPW + gsub < sp ? b0 + q * GPW + gsub : b0];
        tsa_wave_sync();
        sp = b0;
        nst++;
#pragma unroll
        for (int q = 0; q < R; q++) {
          if (q * GPW >= k) break;
          const bool in = q * GPW + gsub < k;
          bool c1 = false, c2 = false;
          uint4 n1{}, n2{};
          if (in) {
            if (tsa_team_has_rule(e[q].x, m)) {
              // (leaves read node 0's words, which are not used)
              uint32_t cO = 0, dO = 0, aO = 0, cM = 0, dM = 0, aM = 0;
              const TsaTeamMove o = tsa_team_visit<W, MODE, false>(
                  P, lab, ch, cc, nullptr, s_lse, s_ilse, T_, e[q], beta, t, [&](int On, int Mn) {
                    const int io = On >= m ? On - m : 0, im = Mn >= m ? Mn - m : 0;
                    cO = ch[io];
                    dO = dr[io];
                    aO = cc.a[io];
                    cM = ch[im];
                    dM = dr[im];
                    aM = cc.a[im];
                  });
              const int l = (int)(o.chv & 0xFFFFu), r = (int)(o.chv >> 16);
              const uint4 eP{o.chp, dr[o.Pn - m], o.cp, (uint32_t)o.Pn};
              const uint4 eX{o.acc ? cM : cO, o.acc ? dM : dO, o.acc ? aM : aO, (uint32_t)(o.acc ? o.Mn : o.On)};
              const bool pl = l == o.Pn;
              n1 = pl ? eP : eX;
              n2 = pl ? eX : eP;
              c1 = t == 0 && l >= m;
              c2 = t == 0 && r >= m;
              if (t == 0) {
                np++;
                na += o.acc;
              }
            }
            if (t == 0) nv++;
          }
          const uint64_t b1 = __ballot(c1), b2 = __ballot(c2);
          int pos = sp + tsa_rank(b1) + tsa_rank(b2);
          if (c2) wl[pos++] = n2;
          if (c1) wl[pos] = n1;
          sp += __popcll(b1) + __popcll(b2);
        }
        tsa_wave_sync();
      }
      __syncthreads();
      if constexpr (LVL) {
        if (--left == 0) {
          if (ev >= 0) {
            keep_costs();
            __syncthreads();
          }
          next_level();
        }
      }
    }
  }
  if constexpr (LVL) {
    if (tracker && lane == 0) {
      F->Lv.own[c] = own.s;
      F->Lv.bslot[c] = own.slot;
    }
  }
  // (every wave passed the last sweep's barrier)
  if (eo.cost) {
    float* const gc = eo.cost + (size_t)c * nint4;
    uint16_t* const gz = eo.z + (size_t)c * nint4;
    for (int i = tid; i < nint; i += NT) {
      gc[i] = cc.cost(i);
      gz[i] = (uint16_t)cc.size(i);
    }
  } else if (eo.lc && wv == 0) {
    const TsaEvalOut x = tsa_fold_finish(
        P, [&](int i) { return cc.size(i); }, nullptr, lf, W, T_, lane & 31,
        tsa_fold_rows([&](int i) { return cc.cost(i); }, nint, T_, lane & 31, -INFINITY, 0, (nint + 31) >> 5));
    if (lane == 0) {
      eo.lc[c] = x.lcost;
      eo.sc[c] = x.sc;
      eo.ns[c] = x.ns;
    }
  }
  if (wv > 0) {
    if (eo.ch) {
      uint32_t* const gch = eo.ch + (size_t)c * nint;
      for (int i = tid - 64; i < nint; i += NT - 64) gch[i] = ch[i];
    }
    for (int i = tid - 64; i < P.chain_words / 2; i += NT - 64)
      reinterpret_cast<uint4*>(g)[i] = reinterpret_cast<const uint4*>(base)[i];
    return;
  }
  const long long sp_ = tsa_wave_sum(np), sa_ = tsa_wave_sum(na), sv_ = tsa_wave_sum(nv);
  if (lane == 0) {  // counters spread over TSA_STAT_SLOTS addresses each, summed by the host
    unsigned long long* st = stats + (c & (TSA_STAT_SLOTS - 1));
    atomicAdd(&st[TSA_ST_PROP * TSA_STAT_SLOTS], (unsigned long long)sp_);
    atomicAdd(&st[TSA_ST_ACC * TSA_STAT_SLOTS], (unsigned long long)sa_);
    atomicAdd(&st[TSA_ST_STEPS * TSA_STAT_SLOTS], (unsigned long long)nst);
    atomicAdd(&st[TSA_ST_VISITS * TSA_STAT_SLOTS], (unsigned long long)sv_);
    atomicAdd(&st[TSA_ST_BUSY * TSA_STAT_SLOTS], (unsigned long long)sv_);
  }
}

template <int W, int MODE, bool LVL>
static hipError_t launch_pre_t(const TsaKParams& P, uint64_t* rec, const uint64_t* leaf, const uint32_t* fix, int nchains,
                               float beta, uint32_t sweep0, int nsweeps, unsigned long long* stats,
                               const TsaEnergyOut& eo, hipStream_t st, hipEvent_t e0, hipEvent_t e1,
                               const TsaLevels* lv, int* res) {
  const size_t smem = (size_t)tsa_team_pre_lds(P.m, P.nint, W, P.chain_words, MODE, 1 + (LVL ? 1 : 0)).bytes;
  const int threads = 64 * (1 + TSA_DRAW_HELPERS);
  const void* const fn = reinterpret_cast<const void*>(&k_team_pre<W, MODE, LVL>);
  if (smem > 65536) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
  }
  if (res) return hipOccupancyMaxActiveBlocksPerMultiprocessor(res, fn, threads, smem);  // a query, no launch
  if (P.chain0 < 0 || P.chain0 >= nchains || eo.blk.n > 0) return hipErrorInvalidValue;
  hipExtLaunchKernelGGL((k_team_pre<W, MODE, LVL>), dim3(nchains - P.chain0), dim3(threads), (uint32_t)smem, st, e0, e1, 0u,
                        P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, lv ? *lv : TsaLevels{});
  return hipGetLastError();
}

bool tsa_team_pre_fits(const TsaKParams& P, int lds_max) {
  return tsa_team_pre_lds(P.m, P.nint, P.W, P.chain_words, 1, 2).bytes <= lds_max - TSA_TEAM_STATIC_LDS;
}

hipError_t tsa_launch_team_pre(int W, int mode, const TsaKParams& P, uint64_t* rec, const uint64_t* leaf,
                               const uint32_t* fix, int nchains, float beta, uint32_t sweep0, int nsweeps,
                               unsigned long long* stats, const TsaEnergyOut& eo, hipStream_t st, hipEvent_t e0,
                               hipEvent_t e1, const TsaLevels* lv, int* res) {
#define TSA_PRE_GO(W, MODE)                                                                                            \
  return lv ? launch_pre_t<W, MODE, true>(P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1, lv, \
                                          res)                                                                         \
            : launch_pre_t<W, MODE, false>(P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, eo, st, e0, e1,   \
                                           lv, res)
#define TSA_PRE_MODES(W)                 \
  if (mode == 0) { TSA_PRE_GO(W, 0); }   \
  if (mode == 1) { TSA_PRE_GO(W, 1); }   \
  TSA_PRE_GO(W, 2)
  switch (W) {
    case 1: TSA_PRE_MODES(1);
    case 2: TSA_PRE_MODES(2);
    case 4: TSA_PRE_MODES(4);
    case 8: TSA_PRE_MODES(8);
    default: return hipErrorInvalidValue;
  }
#undef TSA_PRE_MODES
#undef TSA_PRE_GO
}
