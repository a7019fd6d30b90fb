// tsa_fold.h -- whole-chain evaluation from per-node costs (device code shared by tsa_kernels.hip and
// tsa_wide.hip).
//
// The reference evaluates a chain with 32 lanes (csrc/treesa_gpu.cu:386-434): lane t computes the cost of
// internal nodes t, t+32, ... and folds them with lse_f from -inf, then an xor butterfly 16, 8, 4, 2, 1
// combines the lanes; sc, the number of internal nodes of maximal size and |S| are integer reductions.
// Node costs do not depend on the fold, so they may be computed by any lanes in any order and held in
// memory; tsa_fold32 then runs the fold in the reference's order and is bit-identical to the one-loop form.
#pragma once
#include "tsa_kernels.h"

struct TsaEvalOut {
  float lcost;
  int sc, sc_int, ncand, ns;
};

// Cost (log2) and masked size Z of internal node i: (left child, right child) -> i, every label set masked
// by ~S (S may be null).  NW = words per label set (W, or P.W when W = 0).
template <int W, int MODE>
__device__ __forceinline__ float tsa_node_eval(const TsaKParams& P, const uint64_t* lab, const uint32_t* ch,
                                               const uint64_t* S, const uint64_t* lf, const TsaMathTabs& T, int i,
                                               int& Zout) {
  const int NW = W > 0 ? W : P.W, m = P.m;
  const uint32_t cw = ch[i];
  const int l = (int)(cw & 0xFFFFu), r = (int)(cw >> 16);
  const uint64_t* x = l >= m ? lab + (size_t)(l - m) * NW : lf + (size_t)l * NW;
  const uint64_t* y = r >= m ? lab + (size_t)(r - m) * NW : lf + (size_t)r * NW;
  const uint64_t* z = lab + (size_t)i * NW;
  int B = 0, M = 0, N = 0, K = 0, Z = 0;
  for (int w = 0; w < NW; w++) {
    const uint64_t nm = S ? ~S[w] : ~0ull;
    const uint64_t zz = z[w] & nm;
    tsa_count3(x[w] & nm, y[w] & nm, zz, B, M, N, K);
    Z += __popcll(zz);
  }
  Zout = Z;
  return tsa_node_cost<MODE>(B, M, N, K, Z, P.model, T);
}

// The 32-lane fold of node costs and masked sizes, cost(i) / size(i) for i in [0, nint) (l32 = lane within a
// 32-lane group; every lane of the group returns the result).  lf / S / NW serve the masked leaf sizes when S is
// set.  The lse chain of a lane is serial; its operands are read TSA_FOLD_BATCH at a time ahead of it, so that no
// step waits on a load, and the size statistics run in a loop of their own.
#define TSA_FOLD_BATCH 8
// Rows [row0, row1) of the serial part: node 32 * row + l32 of each row folded into acc (from -inf, which row 0 starts
// from, lse gives the cost itself).
template <class FC>
__device__ __forceinline__ float tsa_fold_rows(FC cost, int nint, const TsaMathTabs& T, int l32, float acc, int row0,
                                               int row1) {
  const int end = 32 * row1 < nint ? 32 * row1 : nint;
  if (row0 == 0) {
    if (l32 < end) acc = cost(l32) + 0.0f;
    row0 = 1;
  }
  for (int i0 = 32 * row0 + l32; i0 < end; i0 += 32 * TSA_FOLD_BATCH) {
    float cb[TSA_FOLD_BATCH];
#pragma unroll
    for (int q = 0; q < TSA_FOLD_BATCH; q++) {
      const int i = i0 + 32 * q;
      cb[q] = i < end ? cost(i) : 0.0f;
    }
#pragma unroll
    for (int q = 0; q < TSA_FOLD_BATCH; q++)
      if (i0 + 32 * q < end) acc = tsa_lse_f(acc, cb[q], T);
  }
  return acc;
}

// The rest of the fold: the size statistics, then the butterfly over the lanes' acc.
template <class FZ>
__device__ __forceinline__ TsaEvalOut tsa_fold_finish(const TsaKParams& P, FZ size, const uint64_t* S,
                                                      const uint64_t* lf, int NW, const TsaMathTabs& T, int l32,
                                                      float acc) {
  const int nint = P.nint, m = P.m;
  int scl = 0, cntl = 0;
  for (int i0 = l32; i0 < nint; i0 += 32 * TSA_FOLD_BATCH) {  // (the sizes read ahead too)
    int zb[TSA_FOLD_BATCH];
#pragma unroll
    for (int q = 0; q < TSA_FOLD_BATCH; q++) {
      const int i = i0 + 32 * q;
      zb[q] = i < nint ? size(i) : -1;
    }
#pragma unroll
    for (int q = 0; q < TSA_FOLD_BATCH; q++) {
      const int Z = zb[q];
      if (Z > scl) {
        scl = Z;
        cntl = 1;
      } else if (Z == scl) {
        cntl++;
      }
    }
  }
  int scmax = scl;
  tsa_lane_butterfly<32>([&](auto o) {
    acc = tsa_lse_f(acc, tsa_lane_xor<decltype(o)::value>(acc), T);
  });
  scmax = tsa_lane_max<32>(scmax);
  int cnt = (scl == scmax) ? cntl : 0, ns = 0;
  if (S)
    for (int w = l32; w < NW; w += 32) ns += __popcll(S[w]);
  cnt = tsa_lane_sum<32>(cnt);
  if (S) ns = tsa_lane_sum<32>(ns);
  int sc = scmax > P.leaf_sc ? scmax : P.leaf_sc;
  if (S && P.leaf_sc > scmax) {  // a leaf may be the largest tensor: masked leaf sizes
    int ll = 0;
    for (int i = l32; i < m; i += 32) {
      int Z = 0;
      for (int w = 0; w < NW; w++) Z += __popcll(lf[(size_t)i * NW + w] & ~S[w]);
      ll = ll > Z ? ll : Z;
    }
    ll = tsa_lane_max<32>(ll);
    sc = scmax > ll ? scmax : ll;
  }
  TsaEvalOut e;
  e.lcost = acc;
  e.sc = sc;
  e.sc_int = scmax;
  e.ncand = cnt;
  e.ns = ns;
  return e;
}

// The whole fold of cost[0..nint) / z[0..nint).  Costs are floats, or (tc mode, whose node costs are integers)
// 16-bit integers converted exactly.
template <typename CT>
__device__ __forceinline__ TsaEvalOut tsa_fold32(const TsaKParams& P, const CT* cost, const uint16_t* z,
                                                 const uint64_t* S, const uint64_t* lf, int NW, const TsaMathTabs& T,
                                                 int l32) {
  const float acc = tsa_fold_rows([&](int i) { return (float)cost[i]; }, P.nint, T, l32, -INFINITY, 0,
                                  (P.nint + 31) / 32);
  return tsa_fold_finish(P, [&](int i) { return (int)z[i]; }, S, lf, NW, T, l32, acc);
}
