// instantiate.hpp -- per-topology kernel instantiation and launcher tables.
#pragma once

#include "ops.hpp"
#include "k_dyn.hpp"
#include "k_crba.hpp"
#include "k_deriv.hpp"
#include "k_kin.hpp"
#include "k_kkt.hpp"
#include "_gen/topologies.inc"

namespace rbd {

inline unsigned gridFor(int64_t B) { return (unsigned)((B + kTile - 1) / kTile); }

// Below about four tiles per CU the sweeps are latency-bound with one wave per tile.
inline int wavesForBatch(int64_t B) {
  const int64_t tiles = (B + kTile - 1) / kTile;
  return tiles >= 1024 ? 1 : tiles >= 512 ? 2 : 4;
}
// a subtree split pays when the busiest wave (trunk included) has well under the whole tree
template<class TP, int G> constexpr bool abaSplitPays() {
  constexpr WaveSplit<TP, G> WS{};
  int trunk = 0, busiest = 0;
  for (int j = 1; j < TP::NJ; ++j) trunk += WS.owner[j] < 0 ? 1 : 0;
  for (int k = 0; k < G; ++k) busiest = WS.load[k] > busiest ? WS.load[k] : busiest;
  return 5 * (trunk + busiest) <= 3 * (TP::NJ - 1) && abaWavesLdsBytes<TP, G>() <= 160 * 1024;
}
// ... and its LDS (sized for 4-byte scalars) fits at the scalar's width
template<class TP, class S, int G> constexpr bool abaSplitPaysFor() {
  return abaSplitPays<TP, G>() && abaWavesLdsBytes<TP, G>() / 4 * (int)sizeof(S) <= 160 * 1024;
}
template<class TP, class S, int G> constexpr bool rneaSplitPaysFor() {
  constexpr WaveSplit<TP, G> WS{};
  int trunk = 0, busiest = 0;
  for (int j = 1; j < TP::NJ; ++j) trunk += WS.owner[j] < 0 ? 1 : 0;
  for (int k = 0; k < G; ++k) busiest = WS.load[k] > busiest ? WS.load[k] : busiest;
  return 5 * (trunk + busiest) <= 3 * (TP::NJ - 1) && rneaWavesLdsBytes<TP, G>() / 4 * (int)sizeof(S) <= 160 * 1024;
}
// Four waves per tile wherever the tree splits (us per call, one wave / four: 18 dofs 30 / 22
// at 512 rows, 53 / 49 at 200,000; 36 dofs 46 / 29, 126 / 99; FP64 295 / 208), but for FP32
// tiles of which fewer than four fit a CU and more than fit the chip: the 60-dof tree 67 / 52
// at 4,096 and 68 / 54 at 16,384, 132 / 160 at 65,536.
template<class TP, class S>
void launchRnea(hipStream_t st, GM, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> a, View<S> out) {
  if constexpr (rneaSplitPaysFor<TP, S, 4>()) {
    constexpr int perCu = 160 * 1024 / (rneaWavesLdsBytes<TP, 4>() / 4 * (int)sizeof(S));
    if ((sizeof(S) == 8 || perCu >= 4 || B <= (int64_t)perCu * 256 * kTile) && gridFits(B / kTile + 1, 4 * kTile)) {
      hipLaunchKernelGGL((k_rnea_waves<TP, S, 4>), dim3(gridFor(B)), dim3(kTile * 4), 0, st, mc, B, q, v, a, out);
      return;
    }
  }
  hipLaunchKernelGGL((k_rnea<TP, S>), dim3(gridFor(B)), dim3(kTile), 0, st, mc, B, q, v, a, out);
}
// RNEA derivatives: the same test, with the LDS of the staged inputs and the 43-float
// subtree slots
template<class TP, int G> constexpr bool rneadSplitPays() {
  constexpr WaveSplit<TP, G> WS{};
  int trunk = 0, busiest = 0;
  for (int j = 1; j < TP::NJ; ++j) trunk += WS.owner[j] < 0 ? 1 : 0;
  for (int k = 0; k < G; ++k) busiest = WS.load[k] > busiest ? WS.load[k] : busiest;
  constexpr int lds = ((TP::T.nq + 2 * TP::T.nv) * kPitch + WS.nslots * kRneadSlot * kTile) * 4;
  return 5 * (trunk + busiest) <= 3 * (TP::NJ - 1) && lds <= 160 * 1024;
}
// waves of one kernel resident per CU with `threads` threads per workgroup (0 if unknown)
inline int residentWaves(const void* kernel, int threads) {
  int blocks = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, threads, 0) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return blocks * (threads / 64);
}
// Waves per tile: chosen from the batch size, and four waves at every size when the four-wave kernel keeps at least twice as many waves
// resident per CU as the one-wave kernel (humanoid: 389 -> 243 registers per lane, one ->
// two waves per SIMD; ABA at 65,536 configurations 67.7 -> 61.7 us).
template<class TP, class S>
void launchAba(hipStream_t st, GM, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> tau, View<S> out) {
  if constexpr (std::is_same_v<S, double>) {
    // FP64: the one-wave kernel spills its per-joint state (twice the registers of FP32);
    // the four-wave split holds it, where the tree splits
    if constexpr (abaSplitPaysFor<TP, S, 4>())
      hipLaunchKernelGGL((k_aba_waves<TP, S, 4>), dim3(gridFor(B)), dim3(kTile * 4), 0, st, mc, B, q, v, tau, out);
    else
      hipLaunchKernelGGL((k_aba<TP, S>), dim3(gridFor(B)), dim3(kTile), 0, st, mc, B, q, v, tau, out);
  } else {
    bool denser = false;
    if constexpr (abaSplitPays<TP, 4>()) {
      static const bool d = [] {
        const int one = residentWaves((const void*)&k_aba<TP, S>, kTile);
        return one > 0 && residentWaves((const void*)&k_aba_waves<TP, S, 4>, kTile * 4) >= 2 * one;
      }();
      denser = d;
    }
    const int waves = denser ? 4 : wavesForBatch(B);
    if constexpr (abaSplitPays<TP, 4>()) {
      if (waves >= 4) {
        hipLaunchKernelGGL((k_aba_waves<TP, S, 4>), dim3(gridFor(B)), dim3(kTile * 4), 0, st, mc, B, q, v, tau, out);
        return;
      }
    }
    if constexpr (abaSplitPays<TP, 2>()) {
      if (waves >= 2) {
        hipLaunchKernelGGL((k_aba_waves<TP, S, 2>), dim3(gridFor(B)), dim3(kTile * 2), 0, st, mc, B, q, v, tau, out);
        return;
      }
    }
    hipLaunchKernelGGL((k_aba<TP, S>), dim3(gridFor(B)), dim3(kTile), 0, st, mc, B, q, v, tau, out);
  }
}
// the tree splits over four waves (the tests above without an algorithm's LDS)
template<class TP> constexpr bool treeSplits() {
  constexpr WaveSplit<TP, 4> WS{};
  int trunk = 0, busiest = 0;
  for (int j = 1; j < TP::NJ; ++j) trunk += WS.owner[j] < 0 ? 1 : 0;
  for (int k = 0; k < 4; ++k) busiest = WS.load[k] > busiest ? WS.load[k] : busiest;
  return 5 * (trunk + busiest) <= 3 * (TP::NJ - 1);
}
template<class TP, class S, int G> constexpr bool crbaSplitPaysFor() {
  return treeSplits<TP>() && crbaWavesLdsBytes<TP, G>() / 4 * (int)sizeof(S) <= 160 * 1024;
}
template<class TP, class SIN, class SC, int G> constexpr bool cholSplitPaysFor() {
  return treeSplits<TP>() && cholWavesLdsBytes<TP, SC, G>() <= 160 * 1024;
}
// CRBA: up to one tile per CU four waves split the tree (humanoid, 16,384: 49 us of kernel on
// two waves, 22 on four writing the factorisation's entries); beyond, two waves per tile
// (output emission split) keep two waves resident per SIMD
template<class TP, class S>
void launchCrba(hipStream_t st, GM, const S* mc, int64_t B, CView<S> q, View<S> M, int upper) {
  if constexpr (crbaSplitPaysFor<TP, S, 4>()) {
    if (B <= 256 * kTile) {
      hipLaunchKernelGGL((k_crba_waves<TP, S, 4>), dim3(gridFor(B)), dim3(kTile * 4), 0, st, mc, B, q, M, upper);
      return;
    }
  }
  if (TP::NJ <= 3)
    hipLaunchKernelGGL((k_crba<TP, S, 1>), dim3(gridFor(B)), dim3(kTile), 0, st, mc, B, q, M, upper);
  else
    hipLaunchKernelGGL((k_crba<TP, S, 2>), dim3(gridFor(B)), dim3(kTile * 2), 0, st, mc, B, q, M, upper);
}
// four waves per tile where that pays (cholops.cpp)
bool cholSplitPaysAt(int nv, bool rows, int64_t B);
template<class TP, class SIN, class SC>
bool launchCholWaves(hipStream_t st, int64_t B, CView<SIN> M, View<SC> U, View<SC> D) {
  if constexpr (cholSplitPaysFor<TP, SIN, SC, 4>()) {
    if (cholSplitPaysAt(TP::T.nv, M.rs == 1, B)) {
      hipLaunchKernelGGL((k_chol_waves<TP, SIN, SC, 4>), dim3(gridFor(B)), dim3(kTile * 4), 0, st, B, M, U, D);
      return true;
    }
  }
  return false;
}
template<class TP, class S> void launchChol(hipStream_t st, GM, int64_t B, CView<S> M, View<double> U, View<double> D) {
  if (launchCholWaves<TP, S, double>(st, B, M, U, D)) return;
  hipLaunchKernelGGL((k_chol<TP, S, double>), dim3(gridFor(B)), dim3(kTile), 0, st, B, M, U, D);
}
// FP32 factor (ABA derivatives, computeMinverse): M staged into LDS first when the batch
// leaves about two tiles per CU or fewer
template<class TP> void launchChol32(hipStream_t st, GM, int64_t B, CView<float> M, View<float> U, View<float> D) {
  if (launchCholWaves<TP, float, float>(st, B, M, U, D)) return;
  const bool staged = (B + kTile - 1) / kTile <= 512;
  if (staged && cholStagedLdsBytes<TP, float>() <= 160 * 1024)
    hipLaunchKernelGGL((k_chol_staged<TP, float, float>), dim3(gridFor(B)), dim3(kTile), 0, st, B, M, U, D);
  else
    hipLaunchKernelGGL((k_chol<TP, float, float>), dim3(gridFor(B)), dim3(kTile), 0, st, B, M, U, D);
}
template<class TP, class S>
void launchCholSolve(hipStream_t st, GM, int64_t B, CView<double> U, CView<double> D, View<S> x) {
  hipLaunchKernelGGL((k_chol64_solve<TP, S>), dim3(gridFor(B)), dim3(kTile), 0, st, B, U, D, x);
}
// RNEA derivatives: with few tiles, 4 waves per tile, each running a share of the subtrees
// (WaveSplit), shorten the critical path
template<class TP, class S>
void launchRneaD(hipStream_t st, GM, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> a, View<S> dq, View<S> dv,
                 View<S> M, int mask, int waves) {
  if (waves <= 0) waves = wavesForBatch(B);
  // (FP64: one wave per tile; the split's LDS, sized for 4-byte scalars, does not fit)
  if constexpr (std::is_same_v<S, float> && rneadSplitPays<TP, 4>()) {
    if (waves >= 2) {
      hipLaunchKernelGGL((k_rnead<TP, S, 4>), dim3(gridFor(B)), dim3(kTile * 4), 0, st, mc, B, q, v, a, dq, dv, M,
                         mask);
      return;
    }
  }
  hipLaunchKernelGGL((k_rnead<TP, S, 1>), dim3(gridFor(B)), dim3(kTile), 0, st, mc, B, q, v, a, dq, dv, M, mask);
}
template<class TP, class S>
void launchAbaDSolve(hipStream_t st, GM, int64_t B, CView<S> U, CView<S> D, View<S> Xq, View<S> Xv, View<S> Minv,
                     int jobBegin) {
  constexpr int CT = SolveTile<S>::CT;
  hipLaunchKernelGGL((k_abad_solve<TP, S>), dim3((unsigned)((B + CT - 1) / CT)), dim3(kTile * kSolveWaves), 0, st, B, U,
                     D, Xq, Xv, Minv, jobBegin);
}


// Outputs by rows.  Runs of a lane's own row while the tiles leave the chip idle: a tile's
// latency counts there, and staging the runs adds to it.  Beyond, staged (us per call, own /
// staged; humanoid, placements and motions: 33 / 35 at 4,096, 36 / 36 at 8,192, 48 / 41 at
// 16,384, 62 / 50 at 30,011, 123 / 80 at 65,536, FP64 40 / 40, 46 / 43, 54 / 47, 85 / 69,
// 209 / 194; arm, one wave per tile, 28 / 30 at 16,384, 31 / 31 at 24,000, 47 / 38 at
// 65,536; Jacobian 25 / 26 at 16,384, 29 / 27 at 24,000, FP64 38 / 43 at 30,011, 65 / 58 at
// 48,000).
// Four waves per tile wherever the tree splits; element by element (batch-fastest) up to
// one tile per CU, or two when only the Jacobian is written: there the stores bound the
// kernel beyond that, and one wave's come in better order (humanoid, one wave / four:
// placements and motions 56 / 36 at 16,384, 60 / 69 at 30,011, Jacobian 33 / 24, 34 / 28).
template<class TP, class S>
void launchKin(hipStream_t st, GM, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> a, View<S> oM, View<S> vo,
               View<S> ao, View<S> J, const KinMask& want) {
  constexpr int G = treeSplits<TP>() ? 4 : 1;
  constexpr int64_t perCu = 256 * kTile;  // configurations of one tile per CU
  auto launch = [&](auto Oc, auto Gc) {
    constexpr KinOut O = KinOut(int(Oc));
    constexpr int g = Gc;
    hipLaunchKernelGGL((k_kin<TP, S, O, g>), dim3(gridFor(B)), dim3(kTile * g), 0, st, mc, B, q, v, a, oM, vo, ao, J,
                       want);
  };
  const bool onlyJ = !oM.p && !vo.p;
  if (kinRows(oM, vo, ao, J) && gridFits(B / kTile + 1, G * kTile)) {
    constexpr int bytes = (kinInScalars<TP>() + kinRunScalars<S, KinOut::kStaged>() * G) * (int)sizeof(S);
    if constexpr (bytes <= 160 * 1024) {
      const int64_t own = G == 1 ? perCu * 3 / 2 : !onlyJ ? perCu / 2 : sizeof(S) == 8 ? perCu * 2 : perCu;
      if (B > own && want.joints == ~0ull && want.columns == ~0ull)
        return launch(IC<(int)KinOut::kStaged>{}, IC<G>{});
    }
    return launch(IC<(int)KinOut::kRuns>{}, IC<G>{});
  }
  if constexpr (G > 1) {
    if (B <= perCu * (onlyJ ? 2 : 1)) return launch(IC<(int)KinOut::kElements>{}, IC<G>{});
  }
  launch(IC<(int)KinOut::kElements>{}, IC<1>{});
}

template<class TP, class S>
void launchKkt(hipStream_t st, GM, int64_t B, CView<double> U, CView<double> D, int nc, CView<S> J, CView<S> tau,
               CView<S> nle, CView<S> gamma, double damping, int mode, double rcoef, const KktProx& prox,
               View<S> ddq, View<S> lam) {
  using K = KktShape<S>;
  hipLaunchKernelGGL((k_kkt<TP, S>), dim3((unsigned)((B + K::T - 1) / K::T)), dim3(64 * K::W), 0, st, B, U, D, nc, J,
                     tau, nle, gamma, damping, mode, rcoef, prox, ddq, lam);
}

template<class TP> TopoOps makeOpsBase() {
  TopoOps o{};
  o.name = TP::name;
  o.njoints = TP::NJ;
  o.parent = TP::parent;
  o.type = TP::type;
  o.nq = TP::T.nq;
  o.nv = TP::T.nv;
  o.compact = TP::T.compact ? 1 : 0;
  return o;
}

// Kernel families, one translation unit each so that a topology's kernels compile in
// parallel.  "dyn" (RNEA, ABA) exists for every topology; the others need a compact
// (DFS-ordered) tree.
template<class TP> void add_dyn(TopoOps& o) {
  o.rnea_f32 = &launchRnea<TP, float>;
  o.rnea_f64 = &launchRnea<TP, double>;
  o.aba_f32 = &launchAba<TP, float>;
  o.aba_f64 = &launchAba<TP, double>;
}
template<class TP> void add_crba(TopoOps& o) {
  o.crba_f32 = &launchCrba<TP, float>;
  o.crba_f64 = &launchCrba<TP, double>;
}
template<class TP> void add_chol(TopoOps& o) {
  o.chol_f32 = &launchChol<TP, float>;
  o.chol_f64 = &launchChol<TP, double>;
  o.cholsolve_f32 = &launchCholSolve<TP, float>;
  o.cholsolve_f64 = &launchCholSolve<TP, double>;
  o.chol32_f32 = &launchChol32<TP>;
  o.nnzU = nnzOf<TP>();
}
template<class TP> void add_rnead(TopoOps& o) {
  o.rnead_f32 = &launchRneaD<TP, float>;
  o.rnead_f64 = &launchRneaD<TP, double>;
}
template<class TP> void add_abads(TopoOps& o) {
  o.abad_solve_f32 = &launchAbaDSolve<TP, float>;
  if constexpr (abadSolveLdsBytes<TP, double>() <= 160 * 1024) o.abad_solve_f64 = &launchAbaDSolve<TP, double>;
}
// (topologies whose staged FP64 factor fits the LDS)
template<class TP> void add_kkt(TopoOps& o) {
  if constexpr (kktLdsBytes<TP, float>() <= 160 * 1024 && kktLdsBytes<TP, double>() <= 160 * 1024) {
    o.kkt_f32 = &launchKkt<TP, float>;
    o.kkt_f64 = &launchKkt<TP, double>;
  }
}
template<class TP> void add_kin(TopoOps& o) {
  o.kin_f32 = &launchKin<TP, float>;
  o.kin_f64 = &launchKin<TP, double>;
}

}  // namespace rbd

// one kernel family of one topology
#define RBD_FILL(NAME, FAM) \
  namespace rbd {           \
  void fill_##NAME##_##FAM(TopoOps& o) { add_##FAM<Topo_##NAME>(o); } \
  }
