// tsa_wide_pre.hip -- pre-order sweeps of wide label sets (runtime width): one workgroup per chain, G lanes per proposal.
//
// A pre-order step visits up to 64 ready nodes (parent already visited) from the top of the work list and pushes their
// internal children (the one-wave kernel's order, so the frontier steps it counts are the same; visits of one frontier
// lie in disjoint subtrees and commute).  On a path-like tree a step is one node, and a sweep a thousand dependent steps:
// what a step costs is latency.  So
//   * a proposal's sets are read by G lanes at once, one or two 16-byte chunks each, where a lane of k_sweep walks all W
//     words of five sets in HBM (32 x 32 lattice, W = 32, 64 chains: 3.3 ms a sweep);
//   * while the frontier fits one wave (64 / G nodes), wave 0 goes on alone with no workgroup barrier; a wider one is
//     shared by all waves;
//   * the children words, the sweep's draws (all made at its start by the whole workgroup) and the work list are in LDS;
//   * the node-cost cache is kept as in k_wide: tc-mode visits do not read the pivot's set, and the energies after the
//     launch are a fold of the cache instead of a pass over every set.
#include "tsa_wide.h"

namespace {

__device__ __forceinline__ void pre_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int G, int MODE>
__global__ void __launch_bounds__(1024) k_wide_pre(TsaKParams P, uint64_t* __restrict__ rec,
                                                   const uint64_t* __restrict__ leaf, const uint32_t* __restrict__ fix,
                                                   int nchains, float beta, uint32_t sweep0, int nsweeps,
                                                   unsigned long long* __restrict__ stats, TsaWideSync sy) {
  // LDS: children words and draws u32[nint4], work list u16[nint4] (tsa_wide_pre_lds bytes; the fold at the end stages
  // costs f32 and sizes u16 there)
  extern __shared__ __align__(16) unsigned char tsa_psm[];
  __shared__ float s_lse[64];
  __shared__ uint64_t s_mt[TSA_MT_WORDS];
  __shared__ uint32_t s_cw[64];  // the step's children words after their visits
  __shared__ int s_sp;
  const int tid = (int)threadIdx.x, NT = (int)blockDim.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = P.m, nint = P.nint, nint4 = (nint + 3) & ~3, NW = P.W, nch = NW >> 1, c = (int)blockIdx.x;
  uint32_t* const ch = reinterpret_cast<uint32_t*>(tsa_psm);
  uint32_t* const draws = ch + nint4;
  uint16_t* const wl = reinterpret_cast<uint16_t*>(draws + nint4);
  uint64_t* const lab = rec + (size_t)c * P.chain_words;
  uint32_t* const gch = reinterpret_cast<uint32_t*>(lab + P.ch_off);
  float* const cst = sy.ncost + (size_t)c * nint4;
  uint16_t* const cz = sy.nz + (size_t)c * nint4;
  if (tid < 64) s_lse[tid] = P.lse[tid];
  tsa_math_stage(s_mt);
  const TsaMathTabs T{s_mt, fix, fix + TSA_LOG2FIX_WORDS, s_mt + 32};
  tsa_copy_inflight<uint32_t, 8>(ch, gch, nint, tid, NT);
  constexpr int GPW = 64 / G;
  const int t = lane & (G - 1), grp = tid / G, ngr = NT / G;
  int np = 0, na = 0, nv = 0, nst = 0;
  auto visit = [&](int j, int b0) {  // entry b0 + j of the work list, by a group
    const int v = wl[b0 + j], vi = v - m;
    const uint32_t chv = ch[vi], d = draws[vi];
    uint32_t cw = chv;
    const int l = (int)(chv & 0xFFFFu), r = (int)(chv >> 16);
    const bool li = l >= m, ri = r >= m;
    if (li || ri) {
      const int b2 = (int)(d & 3u);
      const int rule = li && ri ? b2 : (li ? b2 >> 1 : 2 + (b2 >> 1));
      const int slotP = tsa_slot_p(rule), slotM = tsa_slot_m(rule);
      const int Pn = slotP ? r : l, On = slotP ? l : r;
      const uint32_t chp = ch[Pn - m];
      const int Mn = slotM ? (int)(chp >> 16) : (int)(chp & 0xFFFFu);
      const int Kn = slotM ? (int)(chp & 0xFFFFu) : (int)(chp >> 16);
      auto set = [&](int n) {
        return reinterpret_cast<const TsaW2*>(n >= m ? lab + (size_t)(n - m) * NW : leaf + (size_t)n * NW);
      };
      const bool acc = wide_visit_dense<G, MODE, false>(P, T, s_lse, nch, t, Pn - m, vi, slotP, slotM, set(v),
                                                        reinterpret_cast<TsaW2*>(lab + (size_t)(Pn - m) * NW), set(On),
                                                        set(Kn), set(Mn), d, beta, cst, cz, nullptr);
      if (acc) {
        cw = slotP ? ((chv & 0xFFFF0000u) | (uint32_t)Mn) : ((chv & 0xFFFFu) | ((uint32_t)Mn << 16));
        if (t == 0) {
          ch[Pn - m] = slotM ? ((chp & 0xFFFFu) | ((uint32_t)On << 16)) : ((chp & 0xFFFF0000u) | (uint32_t)On);
          ch[vi] = cw;
        }
      }
      if (t == 0) {
        np++;
        na += acc;
      }
    }
    if (t == 0) {
      s_cw[j] = cw;
      nv++;
    }
  };
  auto push = [&](int k, int b0) {  // the internal children of the step's k nodes, by wave 0; the list's new length
    const uint32_t cw = lane < k ? s_cw[lane] : 0u;
    const bool c1 = (int)(cw & 0xFFFFu) >= m, c2 = (int)(cw >> 16) >= m;  // (leaf id 0 beyond the step)
    const uint64_t b1 = __ballot(c1), b2 = __ballot(c2);
    int pos = b0 + tsa_rank(b1) + tsa_rank(b2);
    if (c2) wl[pos++] = (uint16_t)(cw >> 16);
    if (c1) wl[pos] = (uint16_t)(cw & 0xFFFFu);
    return b0 + __popcll(b1) + __popcll(b2);
  };
  for (int s = 0; s < nsweeps; s++) {
    const uint32_t sw = sweep0 + (uint32_t)s;
    __syncthreads();
    for (int i = tid; i < nint; i += NT) {
      const TsaU4 r = tsa_philox(TsaU4{(uint32_t)(m + i), sw, (uint32_t)c, 0u}, P.key0, P.key1);
      draws[i] = (r.y & 0xFFFFFF00u) | (r.x >> 30);  // the uniform's 24 bits above the rule's two
    }
    if (tid == 0) {
      wl[0] = (uint16_t)(2 * m - 2);
      s_sp = 1;
    }
    __syncthreads();
    int sp = 1;
    for (;;) {
      if (wv == 0) {
        while (sp > 0 && sp <= GPW) {  // the whole frontier in this wave's groups
          const int k = sp;
          if (grp < k) visit(grp, 0);
          pre_wave_sync();
          nst++;
          sp = push(k, 0);
          pre_wave_sync();
        }
        if (lane == 0) s_sp = sp;
      }
      __syncthreads();
      sp = s_sp;
      if (sp == 0) break;
      const int k = sp < 64 ? sp : 64, b0 = sp - k;
      for (int j = grp; j < k; j += ngr) visit(j, b0);
      __syncthreads();
      if (wv == 0) {
        nst++;
        sp = push(k, b0);
        pre_wave_sync();
      }
    }
  }
  __syncthreads();
  for (int i = tid; i < nint; i += NT) gch[i] = ch[i];
  if (sy.snap_ch) {  // the level's snapshot: the tree, and the node costs unless this launch folds them
    uint32_t* const sch = sy.snap_ch + (size_t)c * nint;
    for (int i = tid; i < nint; i += NT) sch[i] = ch[i];
    if (sy.snap_cost) {
      const size_t cb = (size_t)c * nint4;
      tsa_copy_inflight<float, 8>(sy.snap_cost + cb, cst, nint, tid, NT);
      tsa_copy_inflight<uint16_t, 8>(sy.snap_nz + cb, cz, nint, tid, NT);
    }
  }
  if (sy.flc) {
    __syncthreads();
    wide_fold(P, c, cst, cz, nullptr, leaf, fix, s_mt, 1, tsa_psm, sy.flc, sy.fsc, sy.fns);
  }
  const long long sp_ = wide_wave_sum(np), sa_ = wide_wave_sum(na), sv_ = wide_wave_sum(nv);
  if (lane == 0) {  // counters spread over TSA_STAT_SLOTS addresses each, summed by the host
    unsigned long long* st = stats + ((c * 16 + wv) & (TSA_STAT_SLOTS - 1));
    atomicAdd(&st[TSA_ST_PROP * TSA_STAT_SLOTS], (unsigned long long)sp_);
    atomicAdd(&st[TSA_ST_ACC * TSA_STAT_SLOTS], (unsigned long long)sa_);
    atomicAdd(&st[TSA_ST_VISITS * TSA_STAT_SLOTS], (unsigned long long)sv_);
    atomicAdd(&st[TSA_ST_BUSY * TSA_STAT_SLOTS], (unsigned long long)sv_);
    if (wv == 0) atomicAdd(&st[TSA_ST_STEPS * TSA_STAT_SLOTS], (unsigned long long)nst);
  }
}

// LDS bytes of k_wide_pre: at least what wide_fold stages (6 B per node).
int tsa_wide_pre_lds(int nint) { return ((nint + 3) & ~3) * 10; }

template <int G, int MODE>
hipError_t launch_pre(int threads, const TsaKParams& P, uint64_t* rec, const uint64_t* leaf, const uint32_t* fix,
                      int nchains, float beta, uint32_t sweep0, int nsweeps, unsigned long long* stats,
                      const TsaWideSync& sy, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  const int smem = tsa_wide_pre_lds(P.nint);
  if (smem > 65536) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_wide_pre<G, MODE>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return e;
  }
  hipExtLaunchKernelGGL((k_wide_pre<G, MODE>), dim3(nchains), dim3(threads), (uint32_t)smem, st, e0, e1, 0u, P, rec, leaf,
                        fix, nchains, beta, sweep0, nsweeps, stats, sy);
  return hipGetLastError();
}

}  // namespace

bool tsa_wide_pre_fits(const TsaKParams& P, int lds_max) {
  return !P.slicing && tsa_wide_pre_lds(P.nint) <= lds_max - 4096 && P.W / 2 <= tsa_wide_cpl(64) * 64;
}

hipError_t tsa_launch_wide_pre(int mode, const TsaKParams& P, uint64_t* rec, const uint64_t* leaf, const uint32_t* fix,
                               int nchains, int ncu, float beta, uint32_t sweep0, int nsweeps,
                               unsigned long long* stats, const TsaWideSync& sy, hipStream_t st, hipEvent_t e0,
                               hipEvent_t e1) {
  const int G = tsa_wide_pre_lanes(P.W), threads = 64 * tsa_wide_pre_waves(nchains, ncu);
#define TSA_PRE_GO(G)                                                                                                    \
  return mode == 0   ? launch_pre<G, 0>(threads, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, sy, st, e0, e1) \
         : mode == 1 ? launch_pre<G, 1>(threads, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, sy, st, e0, e1) \
                     : launch_pre<G, 2>(threads, P, rec, leaf, fix, nchains, beta, sweep0, nsweeps, stats, sy, st, e0, e1)
  switch (G) {
    case 16: TSA_PRE_GO(16);
    case 32: TSA_PRE_GO(32);
    default: TSA_PRE_GO(64);
  }
#undef TSA_PRE_GO
}
