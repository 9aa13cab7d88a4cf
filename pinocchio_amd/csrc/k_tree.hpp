// k_tree.hpp -- tree-parallel kernels: a small tile of configurations per workgroup, the
// joints of the tree, the dofs and the matrix entries spread over its lanes.
//
// The lane-per-configuration kernels walk the whole tree in every lane, so a call takes
// the time of one serial walk however small the batch is, and they write a matrix output
// one scalar per lane, which in the one-configuration-per-row layout touches 64 cache
// lines per store.  Here a workgroup owns kTreeT configurations; its threads are workers
// of kTreeT lanes each (lane b of a worker: configuration b0 + b).  What bounds such a
// workgroup is the chain of dependent LDS accesses, so every phase is as flat as its
// mathematics allows and there are few of them: joint transforms of all joints at once,
// placements by composing over ancestors 1, 2, 4, ... levels up, sums over a subtree
// (a contiguous index range in depth-first numbering) or a path instead of a walk, one
// pass over the columns or the entries of a matrix.  All state is in LDS,
// [slot][configuration]; a matrix leaves from LDS in runs that are contiguous in the
// caller's layout.
//
// The tree is data (one set of kernels for every depth-first numbered tree); formulations
// are those of k_crba.hpp and k_deriv.hpp (world frame with its origin at the floating
// base; crba.hxx:20-99, 498-548; rnea-derivatives.hxx:242-541).
#pragma once

#include "k_deriv.hpp"
#include "k_dyn.hpp"

namespace rbd {
constexpr int kTreeT = 8;            // configurations per workgroup: 8 workers per wave
constexpr int kTreeMaxThreads = 512;

// Device tables of one model's tree: 16-bit entries, staged in LDS by every workgroup.
// The strictly upper entries of the tree pattern are packed by rows: the dofs below dof r
// are r + 1 .. r + sub[r] - 1, so entry (r, c) sits at rp[r] + c.  Offsets into tab:
struct TProg {
  const int16_t* tab;
  int nTabDyn, nTab, nTabFactor;  // entries RNEA and ABA need; and the matrices; and the factor
  int oJLvl, oJList;      // joints by level of the tree
  int oKidP, oKid;        // children of each joint
  int oJump;              // nlog x nj: the ancestor 2^k joints up (0: none)
  int oSubJ;              // per joint: joints of its subtree
  int oDofJ, oDl, oRp, oSub;  // per dof: joint, number of ancestor dofs, rp, subtree dofs
  int oCp, oPat;          // ancestors a of dof c, root first: pairs (a, rp[a]) from pat[2 cp[c]]
  int oLvl, oItems;       // treeFactor: first item of each phase by segment level; the items
  int oFSeg, nslev;       // its segments (first dof, length) and their levels
  int oPairs;             // (r | c << 8) of the entries with r <= c; read from memory
  int oSeg, nseg;         // chain segments: first dof and length (up to four consecutive dofs)
  int oCommon;            // bytes, nv x nv: number of common strict ancestors of r and c; from memory
  int nj, nq, nv, nlev, nlog, nnz;
  uint32_t nvMagic;       // ceil(2^32 / nv): e / nv by multiplication for e < 2^16
};
enum : int { TJ_PARENT = 0, TJ_TYPE, TJ_IQ, TJ_IV, TJ_NV, TJ_REC };

// one record of LDS state: slot k of this lane's configuration at p[k * kTreeT]
template<class S> struct TRec {
  S* p;
  template<class V> __device__ __forceinline__ V get(int k0) const {
    V o;
    S* f = reinterpret_cast<S*>(&o);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(V) / sizeof(S)); ++k) f[k] = p[(k0 + k) * kTreeT];
    return o;
  }
  template<class V> __device__ __forceinline__ void put(int k0, const V& o) const {
    const S* f = reinterpret_cast<const S*>(&o);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(V) / sizeof(S)); ++k) p[(k0 + k) * kTreeT] = f[k];
  }
};
template<class V, class S> __device__ __forceinline__ V ldsConst(const S* p) {
  V o;
  S* f = reinterpret_cast<S*>(&o);
#pragma unroll
  for (int k = 0; k < (int)(sizeof(V) / sizeof(S)); ++k) f[k] = p[k];
  return o;
}
struct __align__(4) TAnc {  // an ancestor dof and its rp
  int16_t a, rp;
};
__device__ __forceinline__ TAnc treeAnc(const TProg& g, const int16_t* tb, int k) {
  return reinterpret_cast<const TAnc*>(tb + g.oPat)[k];
}
// this thread's configuration and worker
__device__ __forceinline__ int treeB() { return threadIdx.x % kTreeT; }
__device__ __forceinline__ int treeW() { return threadIdx.x / kTreeT; }
__device__ __forceinline__ int treeNW() { return blockDim.x / kTreeT; }

// This workgroup's tile.  Workgroups go round robin over the 8 XCDs: consecutive tiles are
// given to one XCD, so that the 32-byte pieces of a batch-fastest row that neighbouring
// tiles write are merged in one L2.  The grid is a multiple of 8; tiles past the last exit.
__device__ __forceinline__ int64_t treeTile() {
  return (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
}

__device__ __forceinline__ void treeStageTab(const TProg& g, int16_t* st, int n) {
  const int32_t* src = reinterpret_cast<const int32_t*>(g.tab);  // padded to whole words
  int32_t* dst = reinterpret_cast<int32_t*>(st);
  for (int e = threadIdx.x; e < (n + 1) / 2; e += blockDim.x) dst[e] = src[e];
}
// n scalars of each joint's constant record from offset o, at dst[j * stride + at]
template<class S, int o, int n, int stride, int at>
__device__ __forceinline__ void treeStageConsts(const S* __restrict__ mc, int nj, S* dst) {
  for (int e = threadIdx.x; e < nj * n; e += blockDim.x) {
    const int j = e / n, k = e - j * n;
    dst[j * stride + at + k] = mc[j * MC_REC + o + k];
  }
}
// rows [0, R) of the tile at dst[k * kTreeT + b]; lanes past the batch end repeat the last
// configuration
template<class S>
__device__ __forceinline__ void treeStage(S* dst, CView<S> g, int R, int64_t b0, int nb) {
  if (g.rs == 1) {
    for (int e = threadIdx.x; e < R * kTreeT; e += blockDim.x) {
      const int b = e / R, k = e - b * R;
      dst[k * kTreeT + b] = g.p[(b0 + (b < nb ? b : nb - 1)) * g.bs + k];
    }
  } else {
    for (int e = threadIdx.x; e < R * kTreeT; e += blockDim.x) {
      const int k = e / kTreeT, b = e % kTreeT;
      dst[e] = g.p[k * g.rs + (b0 + (b < nb ? b : nb - 1)) * g.bs];
    }
  }
}

// rotAbout with the axis per lane (a wave's joints differ): selects, no branches
template<class S> __device__ __forceinline__ void turnRow(S& m0, S& m1, S& m2, int ax, S s, S c) {
  const S a = ax == 0 ? m1 : (ax == 1 ? m2 : m0), b = ax == 0 ? m2 : (ax == 1 ? m0 : m1);
  const S na = c * a + s * b, nb = c * b - s * a;
  const S r0 = ax == 0 ? m0 : (ax == 1 ? nb : na);
  const S r1 = ax == 0 ? na : (ax == 1 ? m1 : nb);
  const S r2 = ax == 0 ? nb : (ax == 1 ? na : m2);
  m0 = r0;
  m1 = r1;
  m2 = r2;
}
// liMi from the staged placement `c` (R row major, p) and this lane's q
template<class S> __device__ __forceinline__ Xform<S> treeJointX(const S* c, int ty, const S* q, int iq) {
  Xform<S> X = ldsConst<Xform<S>>(c);
  if (ty == JT_FF) {
    const S* x = q + iq * kTreeT;
    return compose(X, Xform<S>{quatToRot(x[3 * kTreeT], x[4 * kTreeT], x[5 * kTreeT], x[6 * kTreeT]),
                               {x[0], x[kTreeT], x[2 * kTreeT]}});
  }
  S sn, cs;
  sincosT(q[iq * kTreeT], &sn, &cs);
  const int ax = ty - JT_RX;
  turnRow(X.R.m00, X.R.m01, X.R.m02, ax, sn, cs);
  turnRow(X.R.m10, X.R.m11, X.R.m12, ax, sn, cs);
  turnRow(X.R.m20, X.R.m21, X.R.m22, ax, sn, cs);
  return X;
}
template<class S> __device__ __forceinline__ Mot<S> treeWorldAxis(const Xform<S>& oM, int ax) {
  const V3<S> w = col(oM.R, ax);
  return {cross(oM.p, w), w};
}

// oMi of every joint into jnt(j)[at ..): transforms of all joints, then nlog rounds of
// composing with what the joint 2^k up holds, between the slots `at` and `alt` of the
// records (12 each).  Returns the slot that holds the result.  `base`: drop the free
// flyers' translation (frame origin at the floating base).
template<class S, int REC>
__device__ __forceinline__ int treePlacements(const TProg& g, const int16_t* tb, const S* sc, int cstride, const S* sq,
                                              S* sj, int at, int alt, bool base) {
  const int b = treeB(), w = treeW();
  auto jnt = [&](int j) { return TRec<S>{sj + j * REC * kTreeT + b}; };
  for (int j = 1 + w; j < g.nj; j += treeNW()) {
    const int ty = tb[j * TJ_REC + TJ_TYPE];
    Xform<S> X = treeJointX(sc + j * cstride, ty, sq + b, tb[j * TJ_REC + TJ_IQ]);
    if (base && ty == JT_FF) X.p = {S(0), S(0), S(0)};
    jnt(j).put(at, X);
  }
  __syncthreads();
  for (int k = 0; k < g.nlog; ++k) {
    for (int j = 1 + w; j < g.nj; j += treeNW()) {
      const int a = tb[g.oJump + k * g.nj + j];
      Xform<S> X = jnt(j).template get<Xform<S>>(at);
      if (a > 0) X = compose(jnt(a).template get<Xform<S>>(at), X);
      jnt(j).put(alt, X);
    }
    __syncthreads();
    const int t = at;
    at = alt;
    alt = t;
  }
  return at;
}

// ---------------------------------------------------------------------------------------
// Packed mass matrix of the tile in LDS: sM[e * kTreeT + b], the strictly upper pattern
// entries by rows, then the diagonal (armature added).  sj: kTreeMassJnt slots per joint
// (two placements; then the world inertia in the one and its subtree sum in the other's
// place), sd: kTreeMassDof per dof (world axis); both odd, so that the workers of a wave
// hit different LDS banks.  sc: placement and body inertia.
// ---------------------------------------------------------------------------------------
constexpr int kTreeMassJnt = 25, kTreeMassDof = 7, kTreeMassC = 23;
template<class S>
__device__ __forceinline__ void treeMass(const TProg& g, const int16_t* tb, const S* sc, const S* sq, S* sj, S* sd,
                                         S* sM, const S* __restrict__ arm) {
  const int b = treeB(), w = treeW();
  auto jnt = [&](int j) { return TRec<S>{sj + j * kTreeMassJnt * kTreeT + b}; };
  auto dof = [&](int c) { return TRec<S>{sd + c * kTreeMassDof * kTreeT + b}; };
  const int at = treePlacements<S, kTreeMassJnt>(g, tb, sc, kTreeMassC, sq, sj, 0, 12, true);
  // -- world axes and inertias
  const int y0 = 12 - at;  // a body's inertia; the subtree's goes to `at`
  for (int j = 1 + w; j < g.nj; j += treeNW()) {
    const int ty = tb[j * TJ_REC + TJ_TYPE], iv = tb[j * TJ_REC + TJ_IV];
    const Xform<S> oM = jnt(j).template get<Xform<S>>(at);
    jnt(j).put(y0, transportUp(oM, ldsConst<CInertia<S>>(sc + j * kTreeMassC + 12)));
    if (ty == JT_FF) {
      for (int k = 0; k < 3; ++k) {
        dof(iv + k).put(0, Mot<S>{col(oM.R, k), {S(0), S(0), S(0)}});
        dof(iv + 3 + k).put(0, treeWorldAxis(oM, k));
      }
    } else {
      dof(iv).put(0, treeWorldAxis(oM, ty - JT_RX));
    }
  }
  __syncthreads();
  // -- composite inertias: component k of joint j summed over its subtree
  for (int it = w; it < (g.nj - 1) * 10; it += treeNW()) {
    const int j = 1 + it / 10, k = it % 10, n = tb[g.oSubJ + j];
    const S* x = sj + (j * kTreeMassJnt + y0 + k) * kTreeT + b;
    S acc = x[0];
#pragma unroll 4
    for (int i = 1; i < n; ++i) acc += x[i * kTreeMassJnt * kTreeT];
    sj[(j * kTreeMassJnt + at + k) * kTreeT + b] = acc;
  }
  __syncthreads();
  // -- columns
  for (int c = w; c < g.nv; c += treeNW()) {
    const Mot<S> J = dof(c).template get<Mot<S>>(0);
    const Frc<S> F = cmul(jnt(tb[g.oDofJ + c]).template get<CInertia<S>>(at), J);
    const int cp = tb[g.oCp + c], na = tb[g.oDl + c];
    sM[(g.nnz + c) * kTreeT + b] = dot(J, F) + arm[c];
#pragma unroll 2
    for (int s = 0; s < na; ++s) {
      const TAnc r = treeAnc(g, tb, cp + s);
      sM[(r.rp + c) * kTreeT + b] = dot(dof(r.a).template get<Mot<S>>(0), F);
    }
  }
  __syncthreads();
}
// scalars of LDS that treeMass needs for its records
__host__ __device__ inline size_t treeMassState(const TProg& g) {
  return (size_t)g.nj * kTreeMassJnt * kTreeT + (size_t)g.nv * kTreeMassDof * kTreeT;
}
// scalars of the space that holds the constants and q first and M (and what the caller
// keeps behind it) later: they are dead before the first entry of M is written.  With the
// pairs' ancestor counts read from memory, not staged, this is a workgroup more per CU
// (CRBA and M^-1 of 10,007 humanoid configurations, FP32: 149 -> 129 us)
inline size_t treeMassSpace(const TProg& g, size_t later) {
  const size_t first = (size_t)g.nj * kTreeMassC + (size_t)g.nq * kTreeT;
  return first > later ? first : later;
}
template<class S>
__device__ __forceinline__ void treeMassTile(const TProg& g, int16_t* tb, int nTab, const S* __restrict__ mc,
                                             CView<S> gq, int64_t b0, int nb, S* state, S* sM) {
  S* sj = state;
  S* sd = sj + g.nj * kTreeMassJnt * kTreeT;
  S* sc = sM;
  S* sq = sc + g.nj * kTreeMassC;
  treeStageTab(g, tb, nTab);
  treeStageConsts<S, MC_R, 12, kTreeMassC, 0>(mc, g.nj, sc);
  treeStageConsts<S, MC_CI, 10, kTreeMassC, 12>(mc, g.nj, sc);
  treeStage(sq, gq, g.nq, b0, nb);
  __syncthreads();
  treeMass<S>(g, tb, sc, sq, sj, sd, sM, mc + g.nj * MC_REC);
}

// ---------------------------------------------------------------------------------------
// Dense outputs: a thread holds element e of all kTreeT configurations.  rs == 1: one store
// per configuration, consecutive lanes on consecutive addresses; otherwise the thread's
// configurations are neighbours in memory, kTreeT scalars at once.
// ---------------------------------------------------------------------------------------
template<class S> constexpr int kTreeV = 16 / sizeof(S);
template<class S> using TreeVec = S __attribute__((ext_vector_type(kTreeV<S>)));
template<class S> struct TreeRow {  // one entry, all configurations
  TreeVec<S> v[kTreeT / kTreeV<S>];
};
template<class S> __device__ __forceinline__ TreeRow<S> treeRow(const S* p) {
  TreeRow<S> r;
#pragma unroll
  for (int u = 0; u < kTreeT / kTreeV<S>; ++u) r.v[u] = reinterpret_cast<const TreeVec<S>*>(p)[u];
  return r;
}
template<class S>
__device__ __forceinline__ void treePut(View<S> g, int e, const TreeRow<S>& x, int64_t b0, int nb) {
  constexpr int V = kTreeV<S>;
  S* dst = g.p + (int64_t)e * g.rs + b0 * g.bs;
  if (g.bs == 1 && nb == kTreeT && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
#pragma unroll
    for (int u = 0; u < kTreeT / V; ++u) reinterpret_cast<TreeVec<S>*>(dst)[u] = x.v[u];
  } else {
#pragma unroll
    for (int b = 0; b < kTreeT; ++b)
      if (b < nb) dst[b * g.bs] = x.v[b / V][b % V];
  }
}

// CRBA
template<class S> size_t treeCrbaLds(const TProg& g) {
  return (size_t)((g.nTab + 7) & ~7) * 2 +
         (treeMassState(g) + treeMassSpace(g, (size_t)(g.nnz + g.nv) * kTreeT)) * sizeof(S);
}
template<class S>
__global__ __launch_bounds__(kTreeMaxThreads) void t_crba(TProg g, const S* __restrict__ mc, int64_t B, CView<S> gq,
                                                       View<S> gM, int upperOnly) {
  extern __shared__ __align__(16) unsigned char t_lds[];
  const int64_t b0 = treeTile() * kTreeT;
  if (b0 >= B) return;
  const int nb = (int)(B - b0 < kTreeT ? B - b0 : kTreeT);
  int16_t* tb = reinterpret_cast<int16_t*>(t_lds);
  S* state = reinterpret_cast<S*>(tb + ((g.nTab + 7) & ~7));
  S* sM = state + treeMassState(g);
  treeMassTile<S>(g, tb, g.nTab, mc, gq, b0, nb, state, sM);
  const int nv = g.nv;
  for (int e = threadIdx.x; e < nv * nv; e += blockDim.x) {
    const int c = __umulhi(e, g.nvMagic), r = e - c * nv;
    const int lo = r < c ? r : c, hi = r < c ? c : r;
    // upper-only: the strict lower triangle is left as it is, but for a joint's own block
    if (upperOnly && r > c && tb[g.oDofJ + r] != tb[g.oDofJ + c]) continue;
    const bool nz = hi < lo + tb[g.oSub + lo];
    TreeRow<S> x{};
    if (nz) x = treeRow(sM + (lo == hi ? g.nnz + lo : tb[g.oRp + lo] + hi) * kTreeT);
    treePut(gM, e, x, b0, nb);
  }
}

// ---------------------------------------------------------------------------------------
// Tree factorisation M = U D U^T of the packed LDS copy (cholesky.hxx:17-62) and W = U^-1
// (same packing: the inverse of a tree factor keeps its pattern).  Dofs are eliminated in
// segments S of up to four consecutive dofs of a chain that branches at its end only, the
// segments of one level of the tree of segments together, from the deepest up:
//   1  A[r][c] -= sum_k A[r][k] A[c][k] / D[k]   rows r above or in S, columns c of S, k below S;
//   2  S itself, in the registers of every row's worker: its own entries of A stay as they
//      are in LDS, its D and W_SS are written by one worker;
//   3  W[S][k] = -W_SS (A[S][k] / D[k] + sum_m A[S][m] / D[m] W[m][k])   k below S, m between.
// 3 of a level reads nothing that 1 of the next writes: one phase.  With W explicit, M^-1 =
// W^T D^-1 W is a sum over ancestors without a chain from row to row.  One level per dof
// instead of per segment (three times the phases, one column per item) took 21 us of a
// tile, triangular sweeps with U 40 us, against 13 (humanoid, FP32).
// Leaves 1 / D in sDi and W in sW.
// ---------------------------------------------------------------------------------------
struct __align__(8) TItem {
  int16_t a, b, c, d;  // 1: rp[r], r, segment, row in S (-1: above);  2: rp[r], segment, -, S itself
};                     // 3: k, segment, first path entry, path length
template<class S> __device__ __forceinline__ S treePartSum(S x, int sh) {  // over 2^sh workers
  const S y = x + __shfl_xor(x, kTreeT);
  x = sh > 0 ? y : x;
  const S z = x + __shfl_xor(x, 2 * kTreeT);
  return sh > 1 ? z : x;
}
template<class S>
__device__ __forceinline__ void treeFactor(const TProg& g, const int16_t* tb, S* sM, S* sDi, S* sW) {
  const int b = treeB(), w = treeW(), NW = treeNW(), nnz = g.nnz;
  const TItem* items = reinterpret_cast<const TItem*>(tb + g.oItems);
  S* M = sM + b;
  S* Di = sDi + b;
  S* W = sW + b;
  auto cols = [&](int seg, int& c0, int& n, int (&rp)[4]) {
    c0 = tb[g.oFSeg + 2 * seg];
    n = tb[g.oFSeg + 2 * seg + 1];
#pragma unroll
    for (int i = 0; i < 4; ++i) rp[i] = tb[g.oRp + c0 + (i < n ? i : 0)];
  };
  for (int l = g.nslev - 1; l >= -1; --l) {
    // items of 1 at this level, then of 3 at the level below
    const int16_t* lv = tb + g.oLvl + 4 * (l + 1);
    const int f0 = lv[0], f1 = lv[1], f2 = lv[2], f3 = lv[3];
    const int nF = f1 - f0, nW = f2 - f1;
    // workers [0, nf) take 1, in whole waves, the following ones 3; few items: shared sums
    const int shF = nF * 8 <= NW ? 2 : (nF * 4 <= NW ? 1 : 0), nf = ((nF << shF) + 7) & ~7;
    const int shW = nf + nW * 4 <= NW ? 2 : (nf + nW * 2 <= NW ? 1 : 0), nw = nf + (nW << shW);
    for (int i0 = 0; i0 < nw; i0 += NW) {  // uniform: every lane takes part in the shuffles
      const int i = i0 + w;
      const bool fac = i < nf;
      const int sh = fac ? shF : shW, parts = 1 << sh, part = i & (parts - 1);
      const int id = fac ? i >> sh : nF + ((i - nf) >> sh);
      const bool on = fac ? id < nF : i < nw;
      S acc[4] = {};
      if (on) {
        const TItem it = items[f0 + id];
        int c0, n, rp[4];
        cols(fac ? it.c : it.b, c0, n, rp);
        if (fac) {
          const S* x = M + it.a * kTreeT;
          const int last = c0 + tb[g.oSub + c0] - 1;
          for (int k = c0 + n + part; k <= last; k += 2 * parts) {
            const int k2 = k + parts <= last ? k + parts : last;
            const S u = x[k * kTreeT] * Di[k * kTreeT];
            const S v = k + parts <= last ? x[k2 * kTreeT] * Di[k2 * kTreeT] : S(0);
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] += u * M[(rp[t] + k) * kTreeT] + v * M[(rp[t] + k2) * kTreeT];
          }
        } else {
          const int k = it.a;
          for (int p = part; p < it.d; p += parts) {
            const TAnc q = treeAnc(g, tb, it.c + p);
            const S u = W[(q.rp + k) * kTreeT] * Di[q.a * kTreeT];
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] += u * M[(rp[t] + q.a) * kTreeT];
          }
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = treePartSum(acc[t], sh);
      if (on && part == 0) {
        const TItem it = items[f0 + id];
        int c0, n, rp[4];
        cols(fac ? it.c : it.b, c0, n, rp);
        if (fac) {
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (t < n && t >= it.d) M[(t == it.d ? nnz + c0 + t : it.a + c0 + t) * kTreeT] -= acc[t];
        } else {
          const int k = it.a;
          const S d = Di[k * kTreeT];
          S v[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = t < n ? acc[t] + M[(rp[t] + k) * kTreeT] * d : S(0);
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            S x = v[t];
#pragma unroll
            for (int o = t + 1; o < 4; ++o) x += o < n ? W[(rp[t] + c0 + o) * kTreeT] * v[o] : S(0);
            if (t < n) W[(rp[t] + k) * kTreeT] = -x;
          }
        }
      }
    }
    __syncthreads();
    if (l < 0) break;
    for (int i = f2 + w; i < f3; i += NW) {
      const TItem it = items[i];
      int c0, n, rp[4];
      cols(it.b, c0, n, rp);
      S a[4], s[4][4], di[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        a[c] = !it.d && c < n ? M[(it.a + c0 + c) * kTreeT] : S(0);
        s[c][c] = c < n ? M[(nnz + c0 + c) * kTreeT] : S(1);
#pragma unroll
        for (int r = 0; r < c; ++r) s[r][c] = c < n ? M[(rp[r] + c0 + c) * kTreeT] : S(0);
      }
#pragma unroll
      for (int c = 3; c >= 0; --c) {
        di[c] = S(1) / s[c][c];
#pragma unroll
        for (int j = 0; j < c; ++j) {
          const S u = s[j][c] * di[c];
          a[j] -= a[c] * u;
#pragma unroll
          for (int r = 0; r <= j; ++r) s[r][j] -= s[r][c] * u;
        }
      }
      if (!it.d) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c < n) M[(it.a + c0 + c) * kTreeT] = a[c];
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c < n) Di[(c0 + c) * kTreeT] = di[c];
        // W_SS: inverse of the unit upper block U = s / D
        S v[4][4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int r = c - 1; r >= 0; --r) {
            S x = s[r][c] * di[c];
#pragma unroll
            for (int m = r + 1; m < c; ++m) x += s[r][m] * di[m] * v[m][c];
            v[r][c] = -x;
            if (c < n) W[(rp[r] + c0 + c) * kTreeT] = -x;
          }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------
// computeMinverse: M of the tile, its factor, W = U^-1, then
//   Minv[r][c] = sum over the common ancestors-or-selves a of W[a][r] W[a][c] / D[a].
// sW overlays the sweep's state, which is dead by then.
// ---------------------------------------------------------------------------------------
template<class S> size_t treeMinvLds(const TProg& g) {
  const size_t state = treeMassState(g), w = (size_t)g.nnz * kTreeT;
  return (size_t)((g.nTabFactor + 7) & ~7) * 2 +
         ((state > w ? state : w) + treeMassSpace(g, (size_t)(g.nnz + 2 * g.nv) * kTreeT)) * sizeof(S);
}
template<class S>
__device__ __forceinline__ TreeRow<S> treeMinvEntry(const TProg& g, const int16_t* tb, const S* sW, const S* sDi, int e) {
  const int c = __umulhi(e, g.nvMagic), r = e - c * g.nv;
  const int lo = r < c ? r : c, hi = r < c ? c : r;
  const int n = reinterpret_cast<const uint8_t*>(g.tab + g.oCommon)[e], cl = tb[g.oCp + lo];
  TreeRow<S> x{};
#pragma unroll 2
  for (int k = 0; k < n; ++k) {
    const TAnc a = treeAnc(g, tb, cl + k);
    const TreeRow<S> p = treeRow(sW + (a.rp + lo) * kTreeT), h = treeRow(sW + (a.rp + hi) * kTreeT),
                     d = treeRow(sDi + a.a * kTreeT);
#pragma unroll
    for (int u = 0; u < kTreeT / kTreeV<S>; ++u) x.v[u] += p.v[u] * (h.v[u] * d.v[u]);
  }
  if (hi < lo + tb[g.oSub + lo]) {  // lo itself
    const TreeRow<S> d = treeRow(sDi + lo * kTreeT);
    TreeRow<S> h = d;
    if (lo != hi) {
      h = treeRow(sW + (tb[g.oRp + lo] + hi) * kTreeT);
#pragma unroll
      for (int u = 0; u < kTreeT / kTreeV<S>; ++u) h.v[u] *= d.v[u];
    }
#pragma unroll
    for (int u = 0; u < kTreeT / kTreeV<S>; ++u) x.v[u] += h.v[u];
  }
  return x;
}
template<class S>
__global__ __launch_bounds__(kTreeMaxThreads) void t_minv(TProg g, const S* __restrict__ mc, int64_t B, CView<S> gq,
                                                       View<S> gX) {
  extern __shared__ __align__(16) unsigned char t_lds[];
  const int64_t b0 = treeTile() * kTreeT;
  if (b0 >= B) return;
  const int nb = (int)(B - b0 < kTreeT ? B - b0 : kTreeT);
  int16_t* tb = reinterpret_cast<int16_t*>(t_lds);
  S* sW = reinterpret_cast<S*>(tb + ((g.nTabFactor + 7) & ~7));
  const size_t state = treeMassState(g), nW = (size_t)g.nnz * kTreeT;
  S* sM = sW + (state > nW ? state : nW);
  S* sDi = sM + (g.nnz + g.nv) * kTreeT;
  treeMassTile<S>(g, tb, g.nTabFactor, mc, gq, b0, nb, sW, sM);
  treeFactor<S>(g, tb, sM, sDi, sW);
  for (int e = threadIdx.x; e < g.nv * g.nv; e += blockDim.x) treePut(gX, e, treeMinvEntry<S>(g, tb, sW, sDi, e), b0, nb);
}

// ---------------------------------------------------------------------------------------
// computeRNEADerivatives of the tile into a workspace of packed tiles, for t_dsolve: tile t
// holds treeWsEntries entries of kTreeT configurations each,
//   dtau_dq: upper entries (r, c), lower entries (c, r) at nnz + (r, c), diagonal; dtau_dv
//   the same; M: upper entries, diagonal.
// World velocities are sums of qd J over a dof's ancestors, gravity-shifted accelerations
// sums of (parent velocity x qd J + qdd J); the composite quantities (inertia, its time
// variation, force: 37 scalars, the variation as its symmetric-transposed block, the
// angular block and the linear momentum that both share) are summed child into parent by
// one worker per component; then one worker per column c emits the column's entries
// (k_deriv.hpp).
// LDS: kTreeRdJnt slots per joint (placements, velocity and acceleration; then the 37) and
// kTreeRdDof per dof (J, dV/dq, dA/dq, dA/dv); two workgroups per CU on the humanoid.
// ---------------------------------------------------------------------------------------
constexpr int kTreeRdJnt = 37, kTreeRdDof = 25;
inline int treeWsEntries(const TProg& g) { return 5 * g.nnz + 3 * g.nv; }
template<class S> size_t treeRneadLds(const TProg& g) {
  return (size_t)((g.nTab + 7) & ~7) * 2 +
         ((size_t)g.nj * (kTreeRdJnt * kTreeT + kTreeMassC) +
          (size_t)(g.nv * kTreeRdDof + g.nq + 2 * g.nv) * kTreeT) * sizeof(S);
}
template<class S>
__global__ __launch_bounds__(kTreeMaxThreads) void t_rnead(TProg g, const S* __restrict__ mc, int64_t B, CView<S> gq,
                                                           CView<S> gv, CView<S> ga, S* __restrict__ ws) {
  extern __shared__ __align__(16) unsigned char t_lds[];
  const int64_t tile = treeTile(), b0 = tile * kTreeT;
  if (b0 >= B) return;
  const int nb = (int)(B - b0 < kTreeT ? B - b0 : kTreeT);
  int16_t* tb = reinterpret_cast<int16_t*>(t_lds);
  S* sj = reinterpret_cast<S*>(tb + ((g.nTab + 7) & ~7));
  S* sd = sj + g.nj * kTreeRdJnt * kTreeT;
  S* sc = sd + g.nv * kTreeRdDof * kTreeT;
  S* sq = sc + g.nj * kTreeMassC;
  S* sv = sq + g.nq * kTreeT;
  S* sa = sv + g.nv * kTreeT;
  const int b = treeB(), w = treeW(), NW = treeNW();
  auto jnt = [&](int j) { return TRec<S>{sj + j * kTreeRdJnt * kTreeT + b}; };
  auto dof = [&](int c) { return TRec<S>{sd + c * kTreeRdDof * kTreeT + b}; };
  treeStageTab(g, tb, g.nTab);
  treeStageConsts<S, MC_R, 12, kTreeMassC, 0>(mc, g.nj, sc);
  treeStageConsts<S, MC_CI, 10, kTreeMassC, 12>(mc, g.nj, sc);
  treeStage(sq, gq, g.nq, b0, nb);
  treeStage(sv, gv, g.nv, b0, nb);
  treeStage(sa, ga, g.nv, b0, nb);
  const S* __restrict__ arm = mc + g.nj * MC_REC;
  const S* __restrict__ gr = arm + g.nv;
  const Mot<S> a0 = {{-gr[0], -gr[1], -gr[2]}, {-gr[3], -gr[4], -gr[5]}};
  __syncthreads();
  const int at = treePlacements<S, kTreeRdJnt>(g, tb, sc, kTreeMassC, sq, sj, 0, 12, true);
  // -- world axes
  for (int c = w; c < g.nv; c += NW) {
    const int j = tb[g.oDofJ + c], ty = tb[j * TJ_REC + TJ_TYPE], k = c - tb[j * TJ_REC + TJ_IV];
    const Xform<S> oM = jnt(j).template get<Xform<S>>(at);
    const int ax = ty == JT_FF ? (k < 3 ? k : k - 3) : ty - JT_RX;
    Mot<S> J = treeWorldAxis(oM, ax);
    if (ty == JT_FF && k < 3) J = {J.a, {S(0), S(0), S(0)}};
    dof(c).put(0, J);
  }
  __syncthreads();
  // world velocity of joint j: the sum of qd J over its last dof and that dof's ancestors
  for (int j = 1 + w; j < g.nj; j += NW) {
    const int c = tb[j * TJ_REC + TJ_IV] + tb[j * TJ_REC + TJ_NV] - 1, cp = tb[g.oCp + c], n = tb[g.oDl + c];
    Mot<S> x = scale(sv[c * kTreeT + b], dof(c).template get<Mot<S>>(0));
#pragma unroll 2
    for (int s = 0; s < n; ++s) {
      const int r = treeAnc(g, tb, cp + s).a;
      x = x + scale(sv[r * kTreeT + b], dof(r).template get<Mot<S>>(0));
    }
    jnt(j).put(24, x);
  }
  __syncthreads();
  for (int c = w; c < g.nv; c += NW) {
    const int p = tb[tb[g.oDofJ + c] * TJ_REC + TJ_PARENT];
    const Mot<S> J = dof(c).template get<Mot<S>>(0);
    Mot<S> x = scale(sa[c * kTreeT + b], J);
    if (p > 0) x = x + crossMM(jnt(p).template get<Mot<S>>(24), scale(sv[c * kTreeT + b], J));
    dof(c).put(18, x);
  }
  __syncthreads();
  for (int j = 1 + w; j < g.nj; j += NW) {
    const int c = tb[j * TJ_REC + TJ_IV] + tb[j * TJ_REC + TJ_NV] - 1, cp = tb[g.oCp + c], n = tb[g.oDl + c];
    Mot<S> x = a0;
#pragma unroll 2
    for (int s = 0; s < n; ++s) x = x + dof(treeAnc(g, tb, cp + s).a).template get<Mot<S>>(18);
    jnt(j).put(30, x + dof(c).template get<Mot<S>>(18));
  }
  __syncthreads();
  // -- column data, composite quantities of the bodies
  for (int c = w; c < g.nv; c += NW) {
    const int j = tb[g.oDofJ + c], p = tb[j * TJ_REC + TJ_PARENT];
    const Mot<S> J = dof(c).template get<Mot<S>>(0), ov = jnt(j).template get<Mot<S>>(24);
    Mot<S> dV = zeroMot<S>(), dA = crossMM(a0, J);
    if (p > 0) {
      const Mot<S> ovp = jnt(p).template get<Mot<S>>(24);
      dV = crossMM(ovp, J);
      dA = crossMM(jnt(p).template get<Mot<S>>(30), J) + crossMM(ovp, dV);
    }
    dof(c).put(6, dV);
    dof(c).put(12, dA);
    dof(c).put(18, crossMM(ov, J) + dV);
  }
  __syncthreads();
  for (int j = 1 + w; j < g.nj; j += NW) {
    const Xform<S> oM = jnt(j).template get<Xform<S>>(at);
    const Mot<S> ov = jnt(j).template get<Mot<S>>(24), oa = jnt(j).template get<Mot<S>>(30);
    const CInertia<S> Y = transportUp(oM, ldsConst<CInertia<S>>(sc + j * kTreeMassC + 12));
    const Frc<S> oh = cmul(Y, ov);
    DY<S> D = inertiaVariation(Y, ov, Frc<S>{{S(0), S(0), S(0)}, oh.a});  // LA = AL^T without oh.l
    jnt(j).put(0, Y);
    jnt(j).put(10, D.LA);
    jnt(j).put(19, D.AA);
    jnt(j).put(28, oh.l);
    jnt(j).put(31, cmul(Y, oa) + crossMF(ov, oh));
  }
  __syncthreads();
  // -- child into parent, last joint first; a chain's running sum stays in a register
  for (int k = w; k < 37; k += NW) {
    S* x = sj + k * kTreeT + b;
    S cur = x[(g.nj - 1) * kTreeRdJnt * kTreeT];
    for (int j = g.nj - 1; j > 1; --j) {
      const int p = tb[j * TJ_REC + TJ_PARENT];
      S next = x[(j - 1) * kTreeRdJnt * kTreeT];
      if (p == j - 1) {
        next += cur;
        x[(j - 1) * kTreeRdJnt * kTreeT] = next;
      } else if (p > 0) {
        x[p * kTreeRdJnt * kTreeT] += cur;
      }
      cur = next;
    }
  }
  __syncthreads();
  // -- columns
  const int nnz = g.nnz, nX = 2 * nnz + g.nv;
  S* out = ws + tile * (int64_t)(5 * nnz + 3 * g.nv) * kTreeT + b;
  auto put = [&](int e, S x) { out[e * kTreeT] = x; };
  for (int c = w; c < g.nv; c += NW) {
    const int j = tb[g.oDofJ + c];
    const CInertia<S> Y = jnt(j).template get<CInertia<S>>(0);
    const R3<S> LA0 = jnt(j).template get<R3<S>>(10);
    const R3<S> Fl = skewM(-jnt(j).template get<V3<S>>(28));
    const DY<S> D = {add(LA0, Fl), add(transpose(LA0), Fl), jnt(j).template get<R3<S>>(19)};
    const Frc<S> of = jnt(j).template get<Frc<S>>(31);
    const ColData<S> C = dof(c).template get<ColData<S>>(0);
    const Frc<S> dFda = cmul(Y, C.J);
    const Frc<S> dFdq = cmul(Y, C.dAdq) + dyMul(D, C.dVdq);
    const Frc<S> dFdv = dyMul(D, C.J) + cmul(Y, C.dAdv);
    const Frc<S> dYtJ = dyMulT(D, C.J);
    const Frc<S> dFdqA = dFdq + crossMF(C.J, of);
    put(2 * nnz + c, dot(C.J, dFdq));
    put(nX + 2 * nnz + c, dot(C.J, dFdv));
    put(2 * nX + nnz + c, dot(C.J, dFda) + arm[c]);
    // entries below the diagonal inside a free flyer's block
    const int c1 = tb[j * TJ_REC + TJ_IV] + tb[j * TJ_REC + TJ_NV], rpc = tb[g.oRp + c];
    for (int c2 = c + 1; c2 < c1; ++c2) {
      const Mot<S> J2 = dof(c2).template get<Mot<S>>(0);
      put(nnz + rpc + c2, dot(J2, dFdq));
      put(nX + nnz + rpc + c2, dot(J2, dFdv));
    }
    const int cp = tb[g.oCp + c], na = tb[g.oDl + c], own = tb[j * TJ_REC + TJ_IV];
    for (int s = 0; s < na; ++s) {
      const TAnc a = treeAnc(g, tb, cp + s);
      const ColData<S> R = dof(a.a).template get<ColData<S>>(0);
      const int e = a.rp + c;
      const bool block = a.a >= own;  // same joint: the term J_c x* of stays out
      put(e, block ? dot(R.J, dFdq) : dot(R.J, dFdqA));
      put(nX + e, dot(R.J, dFdv));
      put(2 * nX + e, dot(R.J, dFda));
      if (!block) {
        put(nnz + e, dot(R.dAdq, dFda) + dot(R.dVdq, dYtJ));
        put(nX + nnz + e, dot(R.dAdv, dFda) + dot(R.J, dYtJ));
      }
    }
  }
}

// ---------------------------------------------------------------------------------------
// ABA-derivative solve on the packed tiles of t_rnead: factor of M, W = U^-1 and M^-1 in
// LDS, then -M^-1 X for X = dtau_dq and dtau_dv.
// Columns go four at a time: a segment of up to four consecutive dofs of one chain
// (TProg::oSeg), so that they are zero outside the same rows, the first dof's ancestors
// and subtree, which alone are staged and summed over.  A worker takes four rows and a
// segment of one X: eight LDS reads for sixteen multiply-adds.  (Two sparse products with W
// are half the multiply-adds, but two phases of short sums each: 45 us of a tile against
// 22, humanoid FP32.)  R segments per round.
// gridDim.y == 3, for batches whose tiles alone leave CUs idle: y = 0, 1 the even and odd
// rounds, y = 2 M^-1 (each repeats the factor).
// LDS: M^-1 [row][row][configuration]; the factor, over which the rounds' X goes.
// ---------------------------------------------------------------------------------------
__host__ __device__ __forceinline__ int treeNB(const TProg& g) { return (g.nv + 3) / 4; }  // rows ib, ib + NB, ..
template<class S> size_t treeSolveLds(const TProg& g, int R) {
  const size_t f = (size_t)(2 * g.nnz + 2 * g.nv) * kTreeT, x = (size_t)R * g.nv * 8 * kTreeT;
  return (size_t)((g.nTabFactor + 7) & ~7) * 2 +
         ((size_t)g.nv * treeNB(g) * 4 * kTreeT + (f > x ? f : x)) * sizeof(S);
}
template<class S>
__global__ __launch_bounds__(kTreeMaxThreads) void t_dsolve(TProg g, int64_t B, const S* __restrict__ ws, View<S> gXq,
                                                            View<S> gXv, View<S> gMinv, int R) {
  extern __shared__ __align__(16) unsigned char t_lds[];
  const int64_t tile = treeTile(), b0 = tile * kTreeT;
  if (b0 >= B) return;
  const int nb = (int)(B - b0 < kTreeT ? B - b0 : kTreeT);
  const int nnz = g.nnz, nv = g.nv, nX = 2 * nnz + nv, NB = treeNB(g), PP = NB * 4 * kTreeT;
  int16_t* tb = reinterpret_cast<int16_t*>(t_lds);
  S* sP = reinterpret_cast<S*>(tb + ((g.nTabFactor + 7) & ~7));
  S* sM = sP + nv * PP;
  S* sDi = sM + (nnz + nv) * kTreeT;
  S* sW = sDi + nv * kTreeT;
  S* sx = sM;
  const int b = treeB(), w = treeW(), NW = treeNW();
  const S* in = ws + tile * (int64_t)(5 * nnz + 3 * nv) * kTreeT;
  // -- stage M
  treeStageTab(g, tb, g.nTabFactor);
  for (int e = threadIdx.x; e < (nnz + nv) * kTreeT; e += blockDim.x) sM[e] = in[2 * nX * kTreeT + e];
  __syncthreads();
  // -- factor
  treeFactor<S>(g, tb, sM, sDi, sW);
  // -- inverse
  const bool all = gridDim.y == 1;
  for (int i = threadIdx.x; i < nv * (nv + 1) / 2; i += blockDim.x) {
    const uint32_t rc = reinterpret_cast<const uint16_t*>(g.tab + g.oPairs)[i];
    const int r = rc & 255, c = rc >> 8;
    const TreeRow<S> x = treeMinvEntry<S>(g, tb, sW, sDi, c * nv + r);
    *reinterpret_cast<TreeRow<S>*>(sP + r * PP + c * kTreeT) = x;
    *reinterpret_cast<TreeRow<S>*>(sP + c * PP + r * kTreeT) = x;
  }
  __syncthreads();
  if (all || blockIdx.y == 2) {
    for (int e = threadIdx.x; e < nv * nv; e += blockDim.x) {
      const int c = __umulhi(e, g.nvMagic), r = e - c * nv;
      treePut(gMinv, e, treeRow(sP + c * PP + r * kTreeT), b0, nb);
    }
    if (!all) return;
  }
  // -- products
  const int step = all ? R : 2 * R;
  for (int s0 = all ? 0 : (int)blockIdx.y * R; s0 < g.nseg; s0 += step) {
    const int ns = g.nseg - s0 < R ? g.nseg - s0 : R;
    // X on the related rows: sx[segment][row][X][column][configuration]
    for (int k = 0; k < ns; ++k) {
      const int c0 = tb[g.oSeg + 2 * (s0 + k)], n = tb[g.oSeg + 2 * (s0 + k) + 1];
      const int dl = tb[g.oDl + c0], cp = tb[g.oCp + c0], nr = dl + tb[g.oSub + c0];
      for (int i = w; i < nr * 8; i += NW) {
        const int idx = i >> 3, m = i & 7, col = m & 3;
        const int r = idx < dl ? treeAnc(g, tb, cp + idx).a : c0 + idx - dl;
        const int c = c0 + (col < n ? col : 0);
        const int lo = r < c ? r : c, hi = r < c ? c : r;
        const int e = lo == hi ? 2 * nnz + lo : (r < c ? 0 : nnz) + tb[g.oRp + lo] + hi;
        sx[((k * nv + idx) * 8 + m) * kTreeT + b] =
            hi < lo + tb[g.oSub + lo] ? in[((m >> 2) * nX + e) * kTreeT + b] : S(0);
      }
    }
    __syncthreads();
    for (int i = w; i < 2 * ns * NB; i += NW) {
      const int kh = i / NB, ib = i - kh * NB, k = kh >> 1, h = kh & 1;
      const int c0 = tb[g.oSeg + 2 * (s0 + k)], n = tb[g.oSeg + 2 * (s0 + k) + 1];
      const int dl = tb[g.oDl + c0], cp = tb[g.oCp + c0], sub = tb[g.oSub + c0];
      const S* x = sx + (k * nv * 8 + h * 4) * kTreeT + b;
      const S* P = sP + ib * kTreeT + b;
      S z[4][4] = {};
      auto add = [&](const S* p) {
        S u[4], y[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) u[t] = p[t * NB * kTreeT];
#pragma unroll
        for (int t = 0; t < 4; ++t) y[t] = x[t * kTreeT];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int o = 0; o < 4; ++o) z[t][o] -= u[t] * y[o];
        x += 8 * kTreeT;
      };
#pragma unroll 2
      for (int p = 0; p < dl; ++p) add(P + treeAnc(g, tb, cp + p).a * PP);
#pragma unroll 2
      for (int p = 0; p < sub; ++p) add(P + (c0 + p) * PP);
      const View<S> out = h ? gXv : gXq;
      S* dst = out.p + (b0 + b) * out.bs;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int o = 0; o < 4; ++o) {
          const int r = ib + t * NB;
          if (b < nb && r < nv && o < n) dst[(int64_t)((c0 + o) * nv + r) * out.rs] = z[t][o];
        }
    }
    __syncthreads();
  }
  // -- end
}

// ---------------------------------------------------------------------------------------
// RNEA and ABA (rnea.hxx:17-161, aba.hxx:79-293; local frames and the re-associated bias of
// k_dyn.hpp).  What does not depend on other joints (transforms, body inertias and forces)
// is one phase over all joints; velocities and accelerations go down and forces and
// articulated inertias up by levels of the tree, a parent adding what its children left in
// their records.  Records: the joint transform (12), then
//   RNEA: v, later the force; a, later the force moved to the parent;
//   ABA (of the transform the rotation only: a revolute joint's translation is a constant):
//   inertia (21) and bias force, later those moved to the parent; v, later the acceleration;
//   the accumulated bias, later U / D; u / D - bias . U / D.  (With this and the
//   smaller space of CRBA, the forward dynamics and mass matrix of 16,384 configurations of a
//   27-dof random tree went from 211 us to 193.)
// One workgroup's sweep is some 20 phases of short work for its few workers per level: two
// waves and a small tile leave room for several workgroups per CU.
// ---------------------------------------------------------------------------------------
constexpr int kTreeDynThreads = 128;  // a level has few joints; 16 workers
constexpr int kTreeDynC = 23;         // staged constants: placement, mass, lever, inertia
constexpr int kTreeRneaJnt = 25, kTreeAbaJnt = 49;
template<class S> size_t treeDynLds(const TProg& g, int rec) {
  return (size_t)((g.nTabDyn + 7) & ~7) * 2 +
         ((size_t)g.nj * (rec * kTreeT + kTreeDynC) + (size_t)(g.nq + 3 * g.nv) * kTreeT) * sizeof(S);
}
template<class S> __device__ __forceinline__ Mot<S> treeJointMot(int ty, const S* x) {  // S x of a joint's slice
  if (ty == JT_FF)
    return {{x[0], x[kTreeT], x[2 * kTreeT]}, {x[3 * kTreeT], x[4 * kTreeT], x[5 * kTreeT]}};
  return axisMot(ty - JT_RX, x[0]);
}
template<class S> struct TreeDyn {  // LDS of a tile
  int16_t* tb;
  S *sj, *sc, *sq, *sv, *sx, *so;
};
// stages the tile's inputs and constants; so: nv rows of output
template<class S>
__device__ __forceinline__ TreeDyn<S> treeDynStage(const TProg& g, unsigned char* lds, int rec,
                                                   const S* __restrict__ mc, CView<S> gq, CView<S> gv, CView<S> gx,
                                                   int64_t b0, int nb) {
  TreeDyn<S> t;
  t.tb = reinterpret_cast<int16_t*>(lds);
  t.sj = reinterpret_cast<S*>(t.tb + ((g.nTabDyn + 7) & ~7));
  t.sc = t.sj + g.nj * rec * kTreeT;
  t.sq = t.sc + g.nj * kTreeDynC;
  t.sv = t.sq + g.nq * kTreeT;
  t.sx = t.sv + g.nv * kTreeT;
  t.so = t.sx + g.nv * kTreeT;
  treeStageTab(g, t.tb, g.nTabDyn);
  treeStageConsts<S, MC_R, 12, kTreeDynC, 0>(mc, g.nj, t.sc);
  treeStageConsts<S, MC_M, 10, kTreeDynC, 12>(mc, g.nj, t.sc);
  treeStage(t.sq, gq, g.nq, b0, nb);
  treeStage(t.sv, gv, g.nv, b0, nb);
  treeStage(t.sx, gx, g.nv, b0, nb);
  __syncthreads();
  return t;
}
template<class S>
__device__ __forceinline__ void treeDynOut(const S* so, View<S> g, int R, int64_t b0, int nb) {
  __syncthreads();
  if (g.rs == 1) {
    for (int e = threadIdx.x; e < R * nb; e += blockDim.x) {
      const int b = e / R, k = e - b * R;
      g.p[(b0 + b) * g.bs + k] = so[k * kTreeT + b];
    }
  } else {
    for (int e = threadIdx.x; e < R * kTreeT; e += blockDim.x) {
      const int k = e / kTreeT, b = e % kTreeT;
      if (b < nb) g.p[k * g.rs + (b0 + b) * g.bs] = so[e];
    }
  }
}
template<class S>
__global__ __launch_bounds__(kTreeDynThreads) void t_rnea(TProg g, const S* __restrict__ mc, int64_t B, CView<S> gq,
                                                          CView<S> gv, CView<S> ga, View<S> gtau) {
  extern __shared__ __align__(16) unsigned char t_lds[];
  const int64_t b0 = treeTile() * kTreeT;
  if (b0 >= B) return;
  const int nb = (int)(B - b0 < kTreeT ? B - b0 : kTreeT);
  const TreeDyn<S> t = treeDynStage(g, t_lds, kTreeRneaJnt, mc, gq, gv, ga, b0, nb);
  const int16_t* tb = t.tb;
  const int b = treeB(), w = treeW(), NW = treeNW();
  const S* __restrict__ arm = mc + g.nj * MC_REC;
  const Mot<S> a0 = mcGravityNeg(arm, g.nv);
  auto jnt = [&](int j) { return TRec<S>{t.sj + j * kTreeRneaJnt * kTreeT + b}; };
  for (int j = 1 + w; j < g.nj; j += NW)
    jnt(j).put(0, treeJointX(t.sc + j * kTreeDynC, tb[j * TJ_REC + TJ_TYPE], t.sq + b, tb[j * TJ_REC + TJ_IQ]));
  for (int l = 0; l < g.nlev; ++l) {
    __syncthreads();
    for (int e = tb[g.oJLvl + l] + w, e1 = tb[g.oJLvl + l + 1]; e < e1; e += NW) {
      const int j = tb[g.oJList + e], p = tb[j * TJ_REC + TJ_PARENT], ty = tb[j * TJ_REC + TJ_TYPE];
      const int iv = tb[j * TJ_REC + TJ_IV];
      const Xform<S> X = jnt(j).template get<Xform<S>>(0);
      const Mot<S> vJ = treeJointMot(ty, t.sv + iv * kTreeT + b);
      Mot<S> v = vJ, a = treeJointMot(ty, t.sx + iv * kTreeT + b);
      if (p > 0) {
        v = v + actInv(X, jnt(p).template get<Mot<S>>(12));
        a = a + actInv(X, jnt(p).template get<Mot<S>>(18));
      } else {
        a = a + actInv(X, a0);
      }
      jnt(j).put(12, v);
      jnt(j).put(18, a + crossMM(v, vJ));
    }
  }
  __syncthreads();
  for (int j = 1 + w; j < g.nj; j += NW) {
    const Body<S> Y = ldsConst<Body<S>>(t.sc + j * kTreeDynC + 12);
    const Mot<S> v = jnt(j).template get<Mot<S>>(12);
    jnt(j).put(12, inertiaMul(Y, jnt(j).template get<Mot<S>>(18)) + crossMF(v, inertiaMul(Y, v)));
  }
  for (int l = g.nlev - 1; l >= 0; --l) {
    __syncthreads();
    for (int e = tb[g.oJLvl + l] + w, e1 = tb[g.oJLvl + l + 1]; e < e1; e += NW) {
      const int j = tb[g.oJList + e], ty = tb[j * TJ_REC + TJ_TYPE], iv = tb[j * TJ_REC + TJ_IV];
      Frc<S> f = jnt(j).template get<Frc<S>>(12);
      for (int k = tb[g.oKidP + j], k1 = tb[g.oKidP + j + 1]; k < k1; ++k)
        f = f + jnt(tb[g.oKid + k]).template get<Frc<S>>(18);
      if (ty == JT_FF) {
#pragma unroll
        for (int k = 0; k < 6; ++k)
          t.so[(iv + k) * kTreeT + b] = comp(f, k) + arm[iv + k] * t.sx[(iv + k) * kTreeT + b];
      } else {
        t.so[iv * kTreeT + b] = comp(f.a, ty - JT_RX) + arm[iv] * t.sx[iv * kTreeT + b];
      }
      if (l > 0) jnt(j).put(18, act(jnt(j).template get<Xform<S>>(0), f));
    }
  }
  treeDynOut(t.so, gtau, g.nv, b0, nb);
}

template<class S>
__global__ __launch_bounds__(kTreeDynThreads) void t_aba(TProg g, const S* __restrict__ mc, int64_t B, CView<S> gq,
                                                         CView<S> gv, CView<S> gt, View<S> gddq) {
  extern __shared__ __align__(16) unsigned char t_lds[];
  const int64_t b0 = treeTile() * kTreeT;
  if (b0 >= B) return;
  const int nb = (int)(B - b0 < kTreeT ? B - b0 : kTreeT);
  const TreeDyn<S> t = treeDynStage(g, t_lds, kTreeAbaJnt, mc, gq, gv, gt, b0, nb);
  const int16_t* tb = t.tb;
  const int b = treeB(), w = treeW(), NW = treeNW();
  const S* __restrict__ arm = mc + g.nj * MC_REC;
  const Mot<S> a0 = mcGravityNeg(arm, g.nv);
  constexpr int kI = 9, kP = 30, kV = 36, kC = 42, kS = 48;  // inertia, force, v, bias, scalar
  auto jnt = [&](int j) { return TRec<S>{t.sj + j * kTreeAbaJnt * kTreeT + b}; };
  // a revolute joint's transform (a free flyer's is used once, at its solve)
  auto jointX = [&](int j) {
    return Xform<S>{jnt(j).template get<R3<S>>(0), ldsConst<V3<S>>(t.sc + j * kTreeDynC + 9)};
  };
  for (int j = 1 + w; j < g.nj; j += NW)
    jnt(j).put(0, treeJointX(t.sc + j * kTreeDynC, tb[j * TJ_REC + TJ_TYPE], t.sq + b, tb[j * TJ_REC + TJ_IQ]).R);
  for (int l = 0; l < g.nlev; ++l) {
    __syncthreads();
    for (int e = tb[g.oJLvl + l] + w, e1 = tb[g.oJLvl + l + 1]; e < e1; e += NW) {
      const int j = tb[g.oJList + e], p = tb[j * TJ_REC + TJ_PARENT], ty = tb[j * TJ_REC + TJ_TYPE];
      const Xform<S> X = jointX(j);
      const Mot<S> vJ = treeJointMot(ty, t.sv + tb[j * TJ_REC + TJ_IV] * kTreeT + b);
      Mot<S> v = vJ;
      if (p > 0) v = v + actInv(X, jnt(p).template get<Mot<S>>(kV));
      Mot<S> c = crossMM(v, vJ);
      if (p > 0) c = c + actInv(X, jnt(p).template get<Mot<S>>(kC));
      jnt(j).put(kV, v);
      jnt(j).put(kC, c);
    }
  }
  __syncthreads();
  for (int j = 1 + w; j < g.nj; j += NW) {
    const Body<S> Y = ldsConst<Body<S>>(t.sc + j * kTreeDynC + 12);
    const Mot<S> v = jnt(j).template get<Mot<S>>(kV);
    jnt(j).put(kP, crossMF(v, inertiaMul(Y, v)));
    jnt(j).put(kI, bodyMatrix(Y));
  }
  for (int l = g.nlev - 1; l >= 0; --l) {
    __syncthreads();
    for (int e = tb[g.oJLvl + l] + w, e1 = tb[g.oJLvl + l + 1]; e < e1; e += NW) {
      const int j = tb[g.oJList + e], p = tb[j * TJ_REC + TJ_PARENT], ty = tb[j * TJ_REC + TJ_TYPE];
      const int iv = tb[j * TJ_REC + TJ_IV];
      Sym6<S> Ia = jnt(j).template get<Sym6<S>>(kI);
      Frc<S> pA = jnt(j).template get<Frc<S>>(kP);
      for (int k = tb[g.oKidP + j], k1 = tb[g.oKidP + j + 1]; k < k1; ++k) {
        const int c = tb[g.oKid + k];
        symAdd(Ia, jnt(c).template get<Sym6<S>>(kI));
        pA = pA + jnt(c).template get<Frc<S>>(kP);
      }
      if (ty == JT_FF) {
        // root free flyer: D = Ia + armature (6x6, FP64 LLT), qdd = D^-1 (tau - pA - Ia a')
        const Mot<S> ap = actInv(treeJointX(t.sc + j * kTreeDynC, ty, t.sq + b, tb[j * TJ_REC + TJ_IQ]), a0);
        const Frc<S> Iap = symMul6(Ia, ap);
        double A[21], x[6];
#pragma unroll
        for (int r = 0; r < 6; ++r) {
#pragma unroll
          for (int c = 0; c <= r; ++c) A[lowIdx(r, c)] = double(sget(Ia, r, c));
          A[lowIdx(r, r)] += double(arm[iv + r]);
          x[r] = double(t.sx[(iv + r) * kTreeT + b]) - double(comp(pA, r)) - double(comp(Iap, r));
        }
        spdSolve6(A, x);
#pragma unroll
        for (int r = 0; r < 6; ++r) t.so[(iv + r) * kTreeT + b] = S(x[r]);
        jnt(j).put(kV, Mot<S>{{ap.l.x + S(x[0]), ap.l.y + S(x[1]), ap.l.z + S(x[2])},
                              {ap.a.x + S(x[3]), ap.a.y + S(x[4]), ap.a.z + S(x[5])}});
      } else {
        const int ax = ty - JT_RX;
        const Frc<S> c3 = symCol(Ia, 3), c4 = symCol(Ia, 4), c5 = symCol(Ia, 5);
        auto sel = [&](S x, S y, S z) { return ax == 0 ? x : (ax == 1 ? y : z); };
        const Frc<S> U = {{sel(c3.l.x, c4.l.x, c5.l.x), sel(c3.l.y, c4.l.y, c5.l.y), sel(c3.l.z, c4.l.z, c5.l.z)},
                          {sel(c3.a.x, c4.a.x, c5.a.x), sel(c3.a.y, c4.a.y, c5.a.y), sel(c3.a.z, c4.a.z, c5.a.z)}};
        const S Dinv = S(1) / (comp(U.a, ax) + arm[iv]);
        const S u = t.sx[iv * kTreeT + b] - comp(pA.a, ax);
        const Frc<S> dd = scale(Dinv, U);
        const Mot<S> c = jnt(j).template get<Mot<S>>(kC);
        t.sj[(j * kTreeAbaJnt + kS) * kTreeT + b] = Dinv * u - dot(c, dd);
        jnt(j).put(kC, dd);
        if (p > 0) {
          symRank1Sub(Ia, U, Dinv);
          const Mot<S> ci = crossMM(jnt(j).template get<Mot<S>>(kV), axisMot(ax, t.sv[iv * kTreeT + b]));
          const Frc<S> pa = pA + symMul6(Ia, ci) + scale(Dinv * u, U);
          const Xform<S> X = jointX(j);
          jnt(j).put(kI, transportUp(X, Ia));
          jnt(j).put(kP, act(X, pa));
        }
      }
    }
  }
  for (int l = 0; l < g.nlev; ++l) {
    __syncthreads();
    for (int e = tb[g.oJLvl + l] + w, e1 = tb[g.oJLvl + l + 1]; e < e1; e += NW) {
      const int j = tb[g.oJList + e], p = tb[j * TJ_REC + TJ_PARENT], ty = tb[j * TJ_REC + TJ_TYPE];
      if (ty == JT_FF) continue;
      const Mot<S> x = actInv(jointX(j), p > 0 ? jnt(p).template get<Mot<S>>(kV) : a0);
      const S qdd = t.sj[(j * kTreeAbaJnt + kS) * kTreeT + b] - dot(x, jnt(j).template get<Frc<S>>(kC));
      t.so[tb[j * TJ_REC + TJ_IV] * kTreeT + b] = qdd;
      jnt(j).put(kV, x + axisMot(ty - JT_RX, qdd));
    }
  }
  treeDynOut(t.so, gddq, g.nv, b0, nb);
}

}  // namespace rbd
