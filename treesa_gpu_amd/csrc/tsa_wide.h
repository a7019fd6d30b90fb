// tsa_wide.h -- what the kernels of wide label sets share: 16-byte chunks, counters packed over a lane group, and the
// dense visit (every chunk of a proposal's sets read by its G lanes).  See tsa_wide.hip.
#pragma once
#include "tsa_kernels.h"
#include "tsa_fold.h"

namespace {

struct alignas(16) TsaW2 {
  uint64_t a, b;
};

// Counters of one proposal as a flat list: |d|, |P|, |X|, then K0..K3 (mode 0) or B0..3, M0..3, N0..3,
// K0..3 (modes 1, 2).
template <int MODE>
struct TsaFlat {
  static constexpr int N = MODE == 0 ? 7 : 19;
  static constexpr int NP = (N + 1) / 2;
};

template <int MODE>
__device__ __forceinline__ void counts_pack(const TsaCounts& c, uint32_t (&a)[TsaFlat<MODE>::NP]) {
  int f[TsaFlat<MODE>::NP * 2];
  f[0] = c.sd;
  f[1] = c.sp;
  f[2] = c.sx;
  if (MODE == 0) {
#pragma unroll
    for (int q = 0; q < 4; q++) f[3 + q] = c.K[q];
    f[7] = 0;
  } else {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      f[3 + q] = c.B[q];
      f[7 + q] = c.M[q];
      f[11 + q] = c.N[q];
      f[15 + q] = c.K[q];
    }
    f[19] = 0;
  }
#pragma unroll
  for (int i = 0; i < TsaFlat<MODE>::NP; i++) a[i] = (uint32_t)f[2 * i] | ((uint32_t)f[2 * i + 1] << 16);
}

template <int MODE>
__device__ __forceinline__ void counts_unpack(const uint32_t (&a)[TsaFlat<MODE>::NP], TsaCounts& c) {
  int f[TsaFlat<MODE>::NP * 2];
#pragma unroll
  for (int i = 0; i < TsaFlat<MODE>::NP; i++) {
    f[2 * i] = (int)(a[i] & 0xFFFFu);
    f[2 * i + 1] = (int)(a[i] >> 16);
  }
  c.sd = f[0];
  c.sp = f[1];
  c.sx = f[2];
  if (MODE == 0) {
#pragma unroll
    for (int q = 0; q < 4; q++) c.K[q] = f[3 + q];
  } else {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      c.B[q] = f[3 + q];
      c.M[q] = f[7 + q];
      c.N[q] = f[11 + q];
      c.K[q] = f[15 + q];
    }
  }
}

// Sum over the G lanes of a group (xor butterfly: every lane ends with the total).  Each packed half
// stays below 2^16: a label set has at most 2 * TSA_WIDE_CPL * 64 * 64 = 16384 labels.
template <int G, int N>
__device__ __forceinline__ void group_sum(uint32_t (&a)[N]) {
  tsa_lane_butterfly<G>([&](auto o) {
#pragma unroll
    for (int i = 0; i < N; i++) a[i] += tsa_lane_xor<decltype(o)::value>(a[i]);
  });
}

__device__ __forceinline__ long long wide_wave_sum(long long x) {
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

// The two node costs a rotation changes: P with children K and O (O in M's slot) and v with children P and M (M in O's
// slot); count3 order is (left child, right child, node).  And P's size.
template <int MODE>
__device__ __forceinline__ void wide_cache_accept(const TsaKParams& P, const TsaMathTabs& T, const TsaCounts& cn, int pi,
                                                  int vi, int slotP, int slotM, float* cst, uint16_t* cz) {
  cst[pi] = tsa_node_cost<MODE>(cn.B[2], slotM ? cn.M[2] : cn.N[2], slotM ? cn.N[2] : cn.M[2], cn.K[2], cn.sx, P.model, T);
  cz[pi] = (uint16_t)cn.sx;
  cst[vi] = tsa_node_cost<MODE>(cn.B[3], slotP ? cn.N[3] : cn.M[3], slotP ? cn.M[3] : cn.N[3], cn.K[3], cn.sd, P.model, T);
}

// A proposal by a group of G lanes (t: lane of the group) that stream every chunk of its label sets: the counts, dE, the
// Metropolis test (ry: the visit's second Philox word) and, when accepted, P's new set and the two node costs and P's
// size in the chain's cache (cst / cz; leader lane).  tc mode takes the costs before the move and P's size from that
// cache (exact: every accept rewrites them, and a sweep starts from a full pass), so P's set is never read.  lab:
// internal label sets; qD .. qM: chunks of D, P, O, K and M; sm: with SLICE the lane's chunks of ~S.  Every lane of the
// group returns the decision.
template <int G, int MODE, bool SLICE>
__device__ __forceinline__ bool wide_visit_dense(const TsaKParams& P, const TsaMathTabs& T, const float* s_lse, int nch,
                                                 int t, int pi, int vi, int slotP, int slotM, const TsaW2* qD,
                                                 TsaW2* qP, const TsaW2* qO, const TsaW2* qK, const TsaW2* qM,
                                                 uint32_t ry, float beta, float* cst, uint16_t* cz, const TsaW2* sm) {
  constexpr bool CACHED = MODE == 0;
  constexpr int CPL = tsa_wide_cpl(G);
  int costP = 0, costV = 0, szP = 0;
  if constexpr (CACHED) {
    costP = (int)cst[pi];
    costV = (int)cst[vi];
    szP = (int)cz[pi];
  }
  TsaCounts cn;
  tsa_counts_zero(cn);
  TsaW2 xx[CPL];  // only X stays live across the energy evaluation
  auto mask = [&](int q) { return SLICE ? sm[q] : TsaW2{~0ull, ~0ull}; };
  if constexpr (CACHED) {  // every load in flight at once
    TsaW2 dd[CPL], oo[CPL], kk[CPL], mm[CPL];
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      const int cc = t + q * G;
      if (cc < nch) {
        dd[q] = qD[cc];
        oo[q] = qO[cc];
        kk[q] = qK[cc];
        mm[q] = qM[cc];
      } else {
        dd[q] = oo[q] = kk[q] = mm[q] = TsaW2{0ull, 0ull};
      }
    }
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      xx[q].a = tsa_xset(kk[q].a, oo[q].a, mm[q].a, dd[q].a);
      xx[q].b = tsa_xset(kk[q].b, oo[q].b, mm[q].b, dd[q].b);
      const TsaW2 n = mask(q);
      tsa_acc_after_tc(cn, kk[q].a & n.a, mm[q].a & n.a, oo[q].a & n.a, dd[q].a & n.a, xx[q].a & n.a);
      tsa_acc_after_tc(cn, kk[q].b & n.b, mm[q].b & n.b, oo[q].b & n.b, dd[q].b & n.b, xx[q].b & n.b);
    }
  } else {
    // chunk by chunk: five sets of CPL chunks and nineteen counters at once do not fit 128 registers (G = 8: 111 of
    // them spilled, here 12; eight levels of 512 chains of a 3-regular graph n=2000 in the gpu mode 11.7 -> 4.6 ms)
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      const int cc = t + q * G;
      xx[q] = TsaW2{0ull, 0ull};
      if (cc < nch) {
        const TsaW2 d = qD[cc], p = qP[cc], o = qO[cc], k = qK[cc], mm = qM[cc], n = mask(q);
        xx[q].a = tsa_xset(k.a, o.a, mm.a, d.a);
        xx[q].b = tsa_xset(k.b, o.b, mm.b, d.b);
        tsa_acc<MODE>(cn, k.a & n.a, mm.a & n.a, p.a & n.a, o.a & n.a, d.a & n.a, xx[q].a & n.a);
        tsa_acc<MODE>(cn, k.b & n.b, mm.b & n.b, p.b & n.b, o.b & n.b, d.b & n.b, xx[q].b & n.b);
      }
    }
  }
  float dE;
  if constexpr (CACHED) {
    uint32_t pk[2] = {(uint32_t)cn.sd | ((uint32_t)cn.sx << 16), (uint32_t)cn.K[2] | ((uint32_t)cn.K[3] << 16)};
    group_sum<G, 2>(pk);
    cn.sd = (int)(pk[0] & 0xFFFFu);
    cn.sx = (int)(pk[0] >> 16);
    cn.K[2] = (int)(pk[1] & 0xFFFFu);
    cn.K[3] = (int)(pk[1] >> 16);
    dE = tsa_energy_tc_cached(costP, costV, szP, cn.sd, cn.sx, cn.K[2], cn.K[3], P.model, s_lse);
  } else {
    uint32_t pk[TsaFlat<MODE>::NP];
    counts_pack<MODE>(cn, pk);
    group_sum<G, TsaFlat<MODE>::NP>(pk);
    counts_unpack<MODE>(pk, cn);
    dE = tsa_energy_from_counts<MODE>(cn, P.model, s_lse, T);
  }
  const bool acc = tsa_metropolis(ry, beta, dE, T.exp2);
  if (acc) {
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      const int cc = t + q * G;
      if (cc < nch) qP[cc] = xx[q];
    }
    if (t == 0) wide_cache_accept<MODE>(P, T, cn, pi, vi, slotP, slotM, cst, cz);
  }
  return acc;
}

// The fold of one chain's cached node costs by the calling workgroup: with stage >= 1 the costs (and with
// stage 2 the log2f summary bitmap) are first copied into the workgroup's LDS at lds (vector copies, all
// loads in flight at once: the fold reads them in a serial chain per lane); lanes 0..31 then fold in the
// reference's order and lane 0 writes lc / sc / ns of chain c.  Every thread of the workgroup calls it.
__device__ __forceinline__ void wide_fold(const TsaKParams& P, int c, const float* cst, const uint16_t* zz,
                                          const uint64_t* S, const uint64_t* leaf, const uint32_t* fix,
                                          const uint64_t* s_mt, int stage, unsigned char* lds, float* lc, int* sc,
                                          int* ns) {
  const int nint4 = (P.nint + 3) & ~3;
  const uint32_t* const gmap = fix + TSA_LOG2FIX_WORDS;
  const uint32_t* map = gmap;
  if (stage) {
    float* const scst = reinterpret_cast<float*>(lds);
    uint16_t* const szz = reinterpret_cast<uint16_t*>(lds + (size_t)nint4 * 4);
    const int n4 = nint4 / 4;
#pragma unroll 4
    for (int i = threadIdx.x; i < n4; i += blockDim.x) {
      const float4 cv = reinterpret_cast<const float4*>(cst)[i];
      const uint2 zv = reinterpret_cast<const uint2*>(zz)[i];
      reinterpret_cast<float4*>(scst)[i] = cv;
      reinterpret_cast<uint2*>(szz)[i] = zv;
    }
    if (stage == 2) {
      uint4* const smap = reinterpret_cast<uint4*>(lds + (((size_t)nint4 * 6 + 15) & ~(size_t)15));
      const uint4* src = reinterpret_cast<const uint4*>(gmap);
#pragma unroll 16
      for (int i = threadIdx.x; i < (int)(TSA_LOG2MAP_WORDS / 4); i += blockDim.x) smap[i] = src[i];
      map = reinterpret_cast<const uint32_t*>(smap);
    }
    __syncthreads();
  }
  if (threadIdx.x < 32) {
    const TsaMathTabs T{s_mt, fix, map, s_mt + 32};
    // two call sites, so that each inlined fold knows whether it reads LDS or global memory
    const TsaEvalOut e = stage ? tsa_fold32(P, reinterpret_cast<const float*>(lds),
                                            reinterpret_cast<const uint16_t*>(lds + (size_t)nint4 * 4), S, leaf, P.W,
                                            T, (int)threadIdx.x)
                               : tsa_fold32(P, cst, zz, S, leaf, P.W, T, (int)threadIdx.x);
    if (threadIdx.x == 0) {
      lc[c] = e.lcost;
      sc[c] = e.sc;
      ns[c] = e.ns;
    }
  }
}

// Slice moves on wide chains (k_wide with SLICE): the LDS of a workgroup's chain beside the sweep's own.
struct WideSlice {
  float* cost;     // node costs and masked sizes of the tree under S, exact
  uint16_t* size;
  float* cost2;    // of a proposed slice set
  uint16_t* size2;
  uint64_t* S;
  uint64_t* S2;
};
__device__ __forceinline__ WideSlice wide_slice_lds(unsigned char* p, int nint, int W) {
  const int nint4 = (nint + 3) & ~3;
  WideSlice s;
  s.S = reinterpret_cast<uint64_t*>(p);
  s.S2 = s.S + W;
  s.cost = reinterpret_cast<float*>(s.S2 + W);
  s.cost2 = s.cost + nint4;
  s.size = reinterpret_cast<uint16_t*>(s.cost2 + nint4);
  s.size2 = s.size + nint4;
  return s;
}

// n-th label (set bit) of A & ~S over W words by one wave (S null: A alone), every lane given the same n: a lane per
// word, so that a set in HBM costs one round trip per 64 words.
__device__ __forceinline__ int wide_nth_label(const uint64_t* A, const uint64_t* S, int W, int n, int lane) {
  for (int w0 = 0; w0 < W; w0 += 64) {
    const int w = w0 + lane;
    const uint64_t a = w < W ? A[w] & (S ? ~S[w] : ~0ull) : 0ull;
    const int x = __popcll(a);
    int y = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(y, o, 64);
      if (lane >= o) y += u;
    }
    const uint64_t hit = __ballot(y - x <= n && n < y);
    if (hit) {
      const int k = __ffsll((unsigned long long)hit) - 1;
      uint64_t b = (uint64_t)__shfl((unsigned long long)a, k, 64);
      for (int r = n - __shfl(y - x, k, 64); r > 0; r--) b &= b - 1;
      return (w0 + k) * 64 + __ffsll((unsigned long long)b) - 1;
    }
    n -= __shfl(y, 63, 64);
  }
  return -1;
}

// Slice moves of one chain by its workgroup (the proposals and floats of tsa_slice_step).  Wave 0 makes a proposal from
// the cached sizes; the workgroup evaluates it -- masking or unmasking a label changes only the nodes whose sets hold
// it, so a node reads one word of three sets and in tc mode adjusts its integers (the float modes recount the nodes
// touched), instead of counting three whole sets of W words; wave 0 folds the current costs in lanes 0-31 and the
// proposed ones in lanes 32-63.  An accepted move swaps the two copies.  Every thread calls it after a barrier; it ends
// with one.  Returns true when an evaluation was made; e (wave 0) is then the chain's as the step leaves it.
template <int MODE>
__device__ __forceinline__ bool wide_slice_step(const TsaKParams& P, const uint64_t* lab, const uint32_t* ch, WideSlice& sl,
                                                const uint64_t* leaf, const TsaMathTabs& T, float beta, uint32_t sw,
                                                uint32_t chain, int (*s_move)[2], int* s_acc, int& nsp, int& nsa,
                                                TsaEvalOut& e) {
  const int tid = (int)threadIdx.x, NT = (int)blockDim.x, lane = tid & 63, nint = P.nint, m = P.m, W = P.W;
  bool evaluated = false;
  for (int j = 0; j < P.slice_moves; j++) {
    const TsaU4 r2 = tsa_philox(TsaU4{0x10001u + 2u * (uint32_t)j, sw, chain, 0u}, P.key0, P.key1);
    if (tid < 64) {
      int scm = 0, ncand = 0, ns = 0;
      for (int i = lane; i < nint; i += 64) {
        const int z = sl.size[i];
        ncand = z > scm ? 1 : ncand + (z == scm);
        scm = z > scm ? z : scm;
      }
      for (int w = lane; w < W; w += 64) ns += __popcll(sl.S[w]);
      const int top = tsa_lane_max<64>(scm);
      ns = tsa_lane_sum<64>(ns);
      ncand = tsa_lane_sum<64>(scm == top ? ncand : 0);
      const TsaU4 r1 = tsa_philox(TsaU4{0x10000u + 2u * (uint32_t)j, sw, chain, 0u}, P.key0, P.key1);
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
          uint64_t b = __ballot(i < nint && sl.size[i < nint ? i : 0] == top);
          const int n = __popcll(b);
          if (rr < n) {
            for (; rr > 0; rr--) b &= b - 1;
            node = b0 + __ffsll((unsigned long long)b) - 1;
          } else {
            rr -= n;
          }
        }
        if (node >= 0) ladd = wide_nth_label(lab + (size_t)node * W, sl.S, W, (int)(r1.z % (uint32_t)top), lane);
      }
      if (type != 0) lrem = wide_nth_label(sl.S, nullptr, W, (int)(r1.w % (uint32_t)ns), lane);
      if (lane == 0) {
        s_move[j & 1][0] = ladd;
        s_move[j & 1][1] = lrem;  // (type 2 without a label to add is a removal, type 0 without one no move)
      }
    }
    __syncthreads();
    const int ladd = s_move[j & 1][0], lrem = s_move[j & 1][1];
    if (ladd < 0 && lrem < 0) continue;  // uniform over the workgroup
    for (int w = tid; w < W; w += NT) {
      uint64_t x = sl.S[w];
      if (ladd >> 6 == w) x |= 1ull << (ladd & 63);
      if (lrem >= 0 && lrem >> 6 == w) x &= ~(1ull << (lrem & 63));
      sl.S2[w] = x;
    }
    if (MODE != 0) __syncthreads();
    for (int i = tid; i < nint; i += NT) {
      const uint32_t cw = ch[i];
      const int l = (int)(cw & 0xFFFFu), r = (int)(cw >> 16);
      const uint64_t* x = l >= m ? lab + (size_t)(l - m) * W : leaf + (size_t)l * W;
      const uint64_t* y = r >= m ? lab + (size_t)(r - m) * W : leaf + (size_t)r * W;
      const uint64_t* z = lab + (size_t)i * W;
      int dz = 0, dk = 0;
      bool touched = false;
      auto label = [&](int lb, int sign) {
        if (lb < 0) return;
        const int w = lb >> 6, b = lb & 63;
        const int xb = (int)(x[w] >> b) & 1, yb = (int)(y[w] >> b) & 1, zb = (int)(z[w] >> b) & 1;
        dz += sign * zb;
        dk += sign * (xb & yb & (zb ^ 1));
        touched |= (xb | yb | zb) != 0;
      };
      label(ladd, -1);  // (not in S before, in S2 after)
      label(lrem, 1);
      float c2 = sl.cost[i];
      int z2 = (int)sl.size[i];
      if (MODE == 0) {
        c2 += (float)(dz + dk);
        z2 += dz;
      } else if (touched) {
        c2 = tsa_node_eval<0, MODE>(P, lab, ch, sl.S2, leaf, T, i, z2);
      }
      sl.cost2[i] = c2;
      sl.size2[i] = (uint16_t)z2;
    }
    __syncthreads();
    nsp++;
    if (tid < 64) {
      const bool hi = lane >= 32;
      const float* const fc = hi ? sl.cost2 : sl.cost;
      const uint16_t* const fz = hi ? sl.size2 : sl.size;
      const TsaEvalOut x =
          tsa_fold_finish(P, [&](int i) { return (int)fz[i]; }, hi ? sl.S2 : sl.S, leaf, W, T, lane & 31,
                          tsa_fold_rows([&](int i) { return fc[i]; }, nint, T, lane & 31, -INFINITY, 0, (nint + 31) / 32));
      const float pen = (float)x.sc > P.model.sc_target ? P.model.sc_weight * ((float)x.sc - P.model.sc_target) : 0.0f;
      const float E = (float)x.ns + x.lcost + pen;
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
      float* const c = sl.cost;
      uint16_t* const z = sl.size;
      uint64_t* const s = sl.S;
      sl.cost = sl.cost2;
      sl.cost2 = c;
      sl.size = sl.size2;
      sl.size2 = z;
      sl.S = sl.S2;
      sl.S2 = s;
    }
  }
  __syncthreads();
  return evaluated;
}

}  // namespace
