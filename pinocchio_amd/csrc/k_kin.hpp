// k_kin.hpp -- batched forward kinematics and joint Jacobians (kinematics.hxx:121-145,
// 209-238; jacobian.hxx:23-62): the pass that RNEA, CRBA and the derivatives open with,
// with its results written out instead of consumed.
//
// One lane per configuration, DFS pre-order over the compile-time tree:
//   oMi = oMi[parent] liMi                                   -> gM (12 per joint: R row major, p)
//   v_i = vJ + liMi^-1 v_parent                              -> gV (6 per joint, local frame)
//   a_i = S qdd + v_i x vJ + liMi^-1 a_parent                -> gA (6 per joint, local frame)
//   J[:, dof] = oMi.act(S_dof)  (WORLD frame)                -> gJ (element r + 6 dof)
// Any output may be absent (null pointer); all outputs leave with nontemporal stores.
#pragma once

#include "k_crba.hpp"
#include "kernels_common.hpp"

namespace rbd {

template<class TP> constexpr int kinLdsRows() { return TP::T.nq + 2 * TP::T.nv; }

// N consecutive scalars in vectors of 16 (placements) or two scalars (motions, columns):
// with one configuration per row a lane's outputs are runs in its own row, a lane apart by
// the row length.  Ordinary stores, so that the L2 completes a line from the runs of
// neighbouring joints: one nontemporal scalar at a time took 952 us where this takes 43
// (humanoid, 30,011 rows, 112 MB; 2.6 TB/s).
template<int N, class S> __device__ __forceinline__ void putRun(S* dst, const S* x) {
  constexpr int V = N == 12 ? 16 / (int)sizeof(S) : 2;
  typedef S Vec __attribute__((ext_vector_type(V)));
#pragma unroll
  for (int k = 0; k < N / V; ++k) {
    Vec v;
#pragma unroll
    for (int u = 0; u < V; ++u) v[u] = x[k * V + u];
    reinterpret_cast<Vec*>(dst)[k] = v;
  }
}
// the outputs are by rows and their runs aligned to putRun's vectors
template<class S> bool kinRows(View<S> M, View<S> V, View<S> A, View<S> J) {
  auto ok = [](const View<S>& g, int n) {
    return !g.p || (g.rs == 1 && g.bs % n == 0 && reinterpret_cast<uintptr_t>(g.p) % (n * sizeof(S)) == 0);
  };
  return ok(M, 16 / sizeof(S)) && ok(V, 2) && ok(A, 2) && ok(J, 2);
}

// kRows: every output that is present passed kinRows.  G > 1: G waves share the tile, each
// running the trunk and its subtrees (WaveSplit); nothing goes back up, so there is nothing
// to hand over.  (Humanoid, 16,384 configurations, placements, motions and Jacobian: 45 us
// on one wave, the serial walk of one tile per CU.)
template<class TP, class S, bool kRows, int G, int W>
__device__ __forceinline__ void kinTile(const S* __restrict__ mc_in, int64_t B, CView<S> gq, CView<S> gv, CView<S> ga,
                                        View<S> gM, View<S> gV, View<S> gA, View<S> gJ, KinMask want,
                                        S* __restrict__ lds) {
  constexpr auto& T = TP::T;
  constexpr int NJ = TP::NJ, NQ = T.nq, NV = T.nv;
  constexpr WaveSplit<TP, G> WS{};
  S* sq = lds;
  S* sv = lds + NQ * kPitch;
  S* sa = lds + (NQ + NV) * kPitch;
  const bool wantV = gV.p != nullptr, wantA = gA.p != nullptr;
  const int64_t b0 = int64_t(blockIdx.x) * kTile;
  const int nb = (int)(B - b0 < kTile ? B - b0 : kTile);
  if constexpr (W == 0) stageIn<NQ>(sq, gq, b0, nb);
  if constexpr (W == 1 % G)
    if (wantV) stageIn<NV>(sv, gv, b0, nb);
  if constexpr (W == 2 % G)
    if (wantA) stageIn<NV>(sa, ga, b0, nb);
  __syncthreads();
  const int L = laneId();
  const int64_t b = b0 + L;
  const bool live = L < nb;

  Xform<S> oM[NJ];
  Mot<S> vj[NJ], aj[NJ];
  // N consecutive rows of an output; kRows: one run of the configuration's memory
  auto put = [&](auto Nc, View<S> g, int row, const S* x) {
    constexpr int N = Nc;
    if (!live) return;
    if constexpr (kRows) {
      putRun<N>(g.p + b * g.bs + row, x);
    } else {
#pragma unroll
      for (int k = 0; k < N; ++k) stOut(&g.p[(int64_t)(row + k) * g.rs + b * g.bs], x[k]);
    }
  };

  static_for<0, NJ - 1>([&](auto K) {
    constexpr int i = TP::T.order[K];
    if constexpr (WS.runs(i, W)) {
    constexpr bool mine = WS.writer(i) == W;
    const bool out = mine && ((want.joints >> i) & 1);
    stepFence();
    const S* __restrict__ mc = stepConsts(mc_in);
    constexpr int p = TP::T.parent[i];
    constexpr int ty = TP::T.type[i];
    constexpr int iq = TP::T.iq[i], iv = TP::T.iv[i], nvi = TP::T.nvj[i];
    Xform<S> X;
    Mot<S> vJ;
    if constexpr (ty == JT_FF) {
      S q7[7];
#pragma unroll
      for (int k = 0; k < 7; ++k) q7[k] = sq[(iq + k) * kPitch + L];
      X = freeflyerX(mc, i, q7, false);
      if (wantV)
        vJ = {{sv[iv * kPitch + L], sv[(iv + 1) * kPitch + L], sv[(iv + 2) * kPitch + L]},
              {sv[(iv + 3) * kPitch + L], sv[(iv + 4) * kPitch + L], sv[(iv + 5) * kPitch + L]}};
    } else {
      S sn, cs;
      sincosT(sq[iq * kPitch + L], &sn, &cs);
      X = revoluteX(mc, i, ty - JT_RX, sn, cs);
      if (wantV) vJ = axisMot(ty - JT_RX, sv[iv * kPitch + L]);
    }
    if constexpr (p > 0) oM[i] = compose(oM[p], X);
    else oM[i] = X;
    if (out && gM.p) {
      const R3<S>& R = oM[i].R;
      const S r12[12] = {R.m00, R.m01, R.m02, R.m10, R.m11, R.m12, R.m20, R.m21, R.m22,
                         oM[i].p.x, oM[i].p.y, oM[i].p.z};
      put(IC<12>{}, gM, (i - 1) * 12, r12);
    }
    if (wantV) {
      Mot<S> vi = vJ;
      if constexpr (p > 0) vi = vi + actInv(X, vj[p]);
      vj[i] = vi;
      const S o[6] = {vi.l.x, vi.l.y, vi.l.z, vi.a.x, vi.a.y, vi.a.z};
      if (out) put(IC<6>{}, gV, (i - 1) * 6, o);
      if (wantA) {
        Mot<S> ai = crossMM(vi, vJ);
        if constexpr (ty == JT_FF) {
          ai = ai + Mot<S>{{sa[iv * kPitch + L], sa[(iv + 1) * kPitch + L], sa[(iv + 2) * kPitch + L]},
                           {sa[(iv + 3) * kPitch + L], sa[(iv + 4) * kPitch + L], sa[(iv + 5) * kPitch + L]}};
        } else {
          ai = ai + axisMot(ty - JT_RX, sa[iv * kPitch + L]);
        }
        if constexpr (p > 0) ai = ai + actInv(X, aj[p]);
        aj[i] = ai;
        const S oa[6] = {ai.l.x, ai.l.y, ai.l.z, ai.a.x, ai.a.y, ai.a.z};
        if (out) put(IC<6>{}, gA, (i - 1) * 6, oa);
      }
    }
    if (mine && gJ.p && ((want.columns >> i) & 1)) {
#pragma unroll
      for (int k = 0; k < nvi; ++k) {
        const Mot<S> c = worldAxis<ty>(oM[i], k);
        const S o[6] = {c.l.x, c.l.y, c.l.z, c.a.x, c.a.y, c.a.z};
        put(IC<6>{}, gJ, (iv + k) * 6, o);
      }
    }
    }
  });
}
template<class TP, class S, bool kRows, int G>
__global__ __launch_bounds__(64 * G) void k_kin(const S* __restrict__ mc, int64_t B, CView<S> gq, CView<S> gv,
                                                CView<S> ga, View<S> gM, View<S> gV, View<S> gA, View<S> gJ,
                                                KinMask want) {
  static_assert(TP::NJ <= 64, "one mask bit per joint");
  __shared__ S lds[kinLdsRows<TP>() * kPitch];
  const int w = G > 1 ? (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  static_for<0, G>([&](auto Wc) {
    constexpr int W = Wc;
    if (w == W) kinTile<TP, S, kRows, G, W>(mc, B, gq, gv, ga, gM, gV, gA, gJ, want, lds);
  });
}

}  // namespace rbd
