// k_kin.hpp -- batched forward kinematics and joint Jacobians (kinematics.hxx:121-145,
// 209-238; jacobian.hxx:23-62): the pass that RNEA, CRBA and the derivatives open with,
// with its results written out instead of consumed.
//
// One lane per configuration, DFS pre-order over the compile-time tree:
//   oMi = oMi[parent] liMi                                   -> gM (12 per joint: R row major, p)
//   v_i = vJ + liMi^-1 v_parent                              -> gV (6 per joint, local frame)
//   a_i = S qdd + v_i x vJ + liMi^-1 a_parent                -> gA (6 per joint, local frame)
//   J[:, dof] = oMi.act(S_dof)  (WORLD frame)                -> gJ (element r + 6 dof)
// Any output may be absent (null pointer).
#pragma once

#include "k_crba.hpp"
#include "kernels_common.hpp"

namespace rbd {

template<class TP> constexpr int kinLdsRows() { return TP::T.nq + 2 * TP::T.nv; }

// N consecutive scalars in vectors of 16 (placements) or two scalars (motions, columns):
// with one configuration per row a lane's outputs are runs in its own row, a lane apart by
// the row length.  Ordinary stores, so that the L2 completes a line from the runs of
// neighbouring joints: one nontemporal scalar at a time took 952 us where this took 47
// (humanoid, placements and motions of 30,011 rows, 86 MB; staged on four waves, below, 31:
// 2.8 TB/s).
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

// How the outputs leave: element by element (any strides), as runs of a lane's own row, or
// as runs through LDS (kRunJoints<S> joints at a time: the wave's lanes write the runs of
// consecutive joints next to each other, so that neighbouring lanes store neighbouring
// vectors of one configuration).  A lane's own runs are a request of the L2 per 8 or 16
// bytes, which bounds the kernel once the tiles fill the chip at any number of waves.
enum class KinOut { kElements, kRuns, kStaged };
template<class S> constexpr int kRunJoints = sizeof(S) == 4 ? 3 : 2;
// Joints whose outputs wave W stores, in groups of consecutive indices: size[i] is the
// group's if joint i is its last, else 0.
template<class TP, int G, int W, int N> struct KinRuns {
  int size[TP::NJ] = {};
  constexpr KinRuns() {
    constexpr auto& T = TP::T;
    constexpr WaveSplit<TP, G> WS{};
    int n = 0, last = -1;
    for (int k = 0; k < TP::NJ - 1; ++k) {
      const int i = T.order[k];
      if (!WS.runs(i, W) || WS.writer(i) != W) continue;
      if (n > 0 && (i != last + 1 || n == N)) {
        size[last] = n;
        n = 0;
      }
      ++n;
      last = i;
    }
    if (n > 0) size[last] = n;
  }
};
// pitch of a configuration's space: whole 16-byte vectors, an odd number of them
template<class S> constexpr int kRunPitch() {
  constexpr int V = 16 / (int)sizeof(S), n = 12 * kRunJoints<S>;
  return n / V % 2 ? n : n + V;
}
// N scalars of each of the wave's configurations from LDS to dst + c bs
template<int N, int V, class S>
__device__ __forceinline__ void flushRuns(const S* st, S* dst, int64_t bs, int nb) {
  typedef S Vec __attribute__((ext_vector_type(V)));
  constexpr int nv = N / V;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int k = 0; k < nv; ++k) {
    const int it = k * kTile + laneId(), c = it / nv, u = it - c * nv;
    if (c < nb)
      *reinterpret_cast<Vec*>(dst + c * bs + u * V) = *reinterpret_cast<const Vec*>(st + c * kRunPitch<S>() + u * V);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// scalars of LDS: the inputs, each wave's space of KinOut::kStaged
template<class TP> constexpr int kinInScalars() { return (kinLdsRows<TP>() * kPitch + 3) / 4 * 4; }
template<class S, KinOut O> constexpr int kinRunScalars() { return O == KinOut::kStaged ? kTile * kRunPitch<S>() : 0; }

// KinOut::kRuns, kStaged: every output that is present passed kinRows; kStaged: all joints
// are wanted.  G > 1: G waves share the tile, each running the trunk and its subtrees
// (WaveSplit); nothing goes back up, so there is nothing to hand over.  (Humanoid, 16,384
// configurations, placements, motions and Jacobian: 45 us on one wave, the serial walk of
// one tile per CU; 14 on four.)
template<class TP, class S, KinOut O, int G, int W>
__device__ __forceinline__ void kinTile(const S* __restrict__ mc_in, int64_t B, CView<S> gq, CView<S> gv, CView<S> ga,
                                        View<S> gM, View<S> gV, View<S> gA, View<S> gJ, KinMask want,
                                        S* __restrict__ lds, S* __restrict__ runs) {
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
  constexpr bool kStaged = O == KinOut::kStaged;
  // N consecutive rows of an output; kRuns: one run of the configuration's memory
  auto put = [&](auto Nc, View<S> g, int row, const S* x) {
    constexpr int N = Nc;
    if (!live) return;
    if constexpr (O == KinOut::kRuns) {
      putRun<N>(g.p + b * g.bs + row, x);
    } else {
#pragma unroll
      for (int k = 0; k < N; ++k) stOut(&g.p[(int64_t)(row + k) * g.rs + b * g.bs], x[k]);
    }
  };
  constexpr KinRuns<TP, G, W, kRunJoints<S>> KR{};
  S* run = runs + L * kRunPitch<S>();

  static_for<0, NJ - 1>([&](auto K) {
    constexpr int i = TP::T.order[K];
    if constexpr (WS.runs(i, W)) {
    constexpr bool mine = WS.writer(i) == W;
    const bool out = !kStaged && mine && (want.joints & KinMask::bit(i));
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
    if (!kStaged && mine && gJ.p && (want.columns & KinMask::bit(i))) {
#pragma unroll
      for (int k = 0; k < nvi; ++k) {
        const Mot<S> c = worldAxis<ty>(oM[i], k);
        const S o[6] = {c.l.x, c.l.y, c.l.z, c.a.x, c.a.y, c.a.z};
        put(IC<6>{}, gJ, (iv + k) * 6, o);
      }
    }
    if constexpr (kStaged && KR.size[i] > 0) {
      constexpr int n = KR.size[i], i0 = i - n + 1;  // the group
      constexpr int d0 = TP::T.iv[i0], nd = iv + nvi - d0;
      if (gM.p) {
        static_for<0, n>([&](auto Jc) {
          constexpr int j = i0 + Jc;
          const R3<S>& R = oM[j].R;
          const S r12[12] = {R.m00, R.m01, R.m02, R.m10, R.m11, R.m12, R.m20, R.m21, R.m22,
                             oM[j].p.x, oM[j].p.y, oM[j].p.z};
          putRun<12>(run + (j - i0) * 12, r12);
        });
        flushRuns<12 * n, 16 / sizeof(S)>(runs, gM.p + b0 * gM.bs + (i0 - 1) * 12, gM.bs, nb);
      }
      auto motions = [&](View<S> g, const Mot<S>* m) {
        static_for<0, n>([&](auto Jc) {
          constexpr int j = i0 + Jc;
          const S o[6] = {m[j].l.x, m[j].l.y, m[j].l.z, m[j].a.x, m[j].a.y, m[j].a.z};
          putRun<6>(run + (j - i0) * 6, o);
        });
        flushRuns<6 * n, 2>(runs, g.p + b0 * g.bs + (i0 - 1) * 6, g.bs, nb);
      };
      if (wantV) motions(gV, vj);
      if (wantA) motions(gA, aj);
      if (gJ.p) {  // a free flyer's columns may take two turns
        constexpr int most = 2 * kRunJoints<S>;
        static_for<0, (nd + most - 1) / most>([&](auto Qc) {
          constexpr int c0 = d0 + Qc * most, nc = d0 + nd - c0 < most ? d0 + nd - c0 : most;
          static_for<0, nc>([&](auto Cc) {
            constexpr int c = c0 + Cc, j = TP::T.dofJoint[c];
            const Mot<S> m = worldAxis<TP::T.type[j]>(oM[j], c - TP::T.iv[j]);
            const S o[6] = {m.l.x, m.l.y, m.l.z, m.a.x, m.a.y, m.a.z};
            putRun<6>(run + Cc * 6, o);
          });
          flushRuns<6 * nc, 2>(runs, gJ.p + b0 * gJ.bs + c0 * 6, gJ.bs, nb);
        });
      }
    }
    }
  });
}
template<class TP, class S, KinOut O, int G>
__global__ __launch_bounds__(64 * G) void k_kin(const S* __restrict__ mc, int64_t B, CView<S> gq, CView<S> gv,
                                                CView<S> ga, View<S> gM, View<S> gV, View<S> gA, View<S> gJ,
                                                KinMask want) {
  constexpr int nIn = kinInScalars<TP>(), nRun = kinRunScalars<S, O>();
  __shared__ __align__(16) S lds[nIn + nRun * G];
  const int w = G > 1 ? (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  static_for<0, G>([&](auto Wc) {
    constexpr int W = Wc;
    if (w == W) kinTile<TP, S, O, G, W>(mc, B, gq, gv, ga, gM, gV, gA, gJ, want, lds, lds + nIn + nRun * W);
  });
}

}  // namespace rbd
