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

namespace rbd {
constexpr int kTreeT = 8;            // configurations per workgroup: 8 workers per wave
constexpr int kTreeMaxThreads = 1024;

// Device tables of one model's tree: 16-bit entries, staged in LDS by every workgroup.
// The strictly upper entries of the tree pattern are packed by rows: the dofs below dof r
// are r + 1 .. r + sub[r] - 1, so entry (r, c) sits at rp[r] + c.  Offsets into tab:
struct TProg {
  const int16_t* tab;
  int nTab, nTabFactor;   // entries without and with the factorisation's lists
  int oJump;              // nlog x nj: the ancestor 2^k joints up (0: none)
  int oSubJ;              // per joint: joints of its subtree
  int oDofJ, oDl, oRp, oSub;  // per dof: joint, number of ancestor dofs, rp, subtree dofs
  int oCp, oPat;          // ancestors a of dof c, root first: pairs (a, rp[a]) from pat[2 cp[c]]
  int oLvl, oItems;       // treeFactor: per dof level the first and first W item; the items
  int oCommon;            // bytes, nv x nv: number of common strict ancestors of r and c
  int nj, nq, nv, nlog, nvlev, nnz;
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
// scalars of LDS that treeMass needs beside sM
inline size_t treeMassState(const TProg& g) {
  return (size_t)g.nj * (kTreeMassJnt * kTreeT + kTreeMassC) + (size_t)g.nv * kTreeMassDof * kTreeT +
         (size_t)g.nq * kTreeT;
}
template<class S>
__device__ __forceinline__ void treeMassTile(const TProg& g, int16_t* tb, int nTab, const S* __restrict__ mc,
                                             CView<S> gq, int64_t b0, int nb, S* state, S* sM) {
  S* sj = state;
  S* sd = sj + g.nj * kTreeMassJnt * kTreeT;
  S* sc = sd + g.nv * kTreeMassDof * kTreeT;
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
  return (size_t)((g.nTab + 7) & ~7) * 2 + (treeMassState(g) + (size_t)(g.nnz + g.nv) * kTreeT) * sizeof(S);
}
template<class S>
__global__ __launch_bounds__(kTreeMaxThreads) void t_crba(TProg g, const S* __restrict__ mc, int64_t B, CView<S> gq,
                                                       View<S> gM, int upperOnly) {
  extern __shared__ __align__(16) unsigned char t_lds[];
  const int64_t b0 = treeTile() * kTreeT;
  if (b0 >= B) return;
  const int nb = (int)(B - b0 < kTreeT ? B - b0 : kTreeT);
  int16_t* tb = reinterpret_cast<int16_t*>(t_lds);
  S* sM = reinterpret_cast<S*>(tb + ((g.nTab + 7) & ~7));
  treeMassTile<S>(g, tb, g.nTab, mc, gq, b0, nb, sM + (g.nnz + g.nv) * kTreeT, sM);
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
// (same packing: the inverse of a tree factor keeps its pattern), by dof level from the
// deepest up.  For a dof j of the level and an ancestor-or-self r (left-looking),
//   A[r][j] = M[r][j] - sum_{k below j} A[r][k] A[j][k] / D[k]       (k = j + 1 .. j + sub[j] - 1),
// and for a dof r of the level and a dof k below it, with the path dofs m between them,
//   W[r][k] = -(A[r][k] / D[k] + sum_m A[r][m] / D[m] W[m][k]).
// Both read deeper levels only, so a level is one phase; where its items are few (the
// trunk, whose sums are long) two or four workers share a sum.  With W explicit, M^-1 =
// W^T D^-1 W and a product with it is a sum over ancestors or descendants without a chain
// from row to row (the triangular sweeps, 36 dependent rows, took 40 us on the humanoid;
// factor and W in two sweeps of levels 29 us).  Leaves D on sM's diagonal, 1 / D in sDi.
// Items: rp[r], rp[j], j, sub[j];  rp[r], k, first path entry, path length.
// ---------------------------------------------------------------------------------------
struct __align__(8) TItem {
  int16_t a, b, c, d;
};
// sum over the 2^sh (1, 2 or 4) neighbouring workers of a wave
template<class S> __device__ __forceinline__ S treePartSum(S x, int sh) {
  const S y = x + __shfl_xor(x, kTreeT);
  x = sh > 0 ? y : x;
  const S z = x + __shfl_xor(x, 2 * kTreeT);
  return sh > 1 ? z : x;
}
template<class S>
__device__ __forceinline__ void treeFactor(const TProg& g, const int16_t* tb, S* sM, S* sDi, S* sW) {
  const int b = treeB(), w = treeW(), NW = treeNW();
  const TItem* items = reinterpret_cast<const TItem*>(tb + g.oItems);
  for (int l = g.nvlev - 1; l >= 0; --l) {
    const int f0 = tb[g.oLvl + 2 * l], f1 = tb[g.oLvl + 2 * l + 1], n = tb[g.oLvl + 2 * l + 2] - f0;
    // workers [0, nf) take the factor's items, in whole waves, the following ones W's
    const int nF = f1 - f0, nW = n - nF;
    const int shF = nF * 8 <= NW ? 2 : (nF * 4 <= NW ? 1 : 0), nf = ((nF << shF) + 7) & ~7;
    const int shW = nf + nW * 4 <= NW ? 2 : (nf + nW * 2 <= NW ? 1 : 0), nw = nf + (nW << shW);
    for (int i0 = 0; i0 < nw; i0 += NW) {  // uniform: every lane takes part in the shuffles
      const int i = i0 + w;
      const bool fac = i < nf;
      const int sh = fac ? shF : shW, parts = 1 << sh, part = i & (parts - 1);
      const int id = fac ? i >> sh : nF + ((i - nf) >> sh);
      const bool on = fac ? id < nF : i < nw;
      const TItem it = items[f0 + (on ? id : 0)];
      const S* x = sM + it.a * kTreeT + b;
      S acc = S(0), m = S(0);
      S* dst;
      // sums in batches of four, the last one filled up with zero weights
      if (fac) {
        const S* y = sM + it.b * kTreeT + b;
        const int j = it.c, last = j + it.d - 1;
        dst = sM + (it.a == it.b ? g.nnz + j : it.a + j) * kTreeT + b;
        m = *dst;
        for (int k = j + 1 + part; k <= last; k += 4 * parts) {
          S u[4], v[4], d[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int kk = k + t * parts <= last ? k + t * parts : last;
            u[t] = x[kk * kTreeT];
            v[t] = y[kk * kTreeT];
            d[t] = sDi[kk * kTreeT + b];
            d[t] = k + t * parts <= last ? d[t] : S(0);
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) acc += u[t] * (v[t] * d[t]);
        }
      } else {
        const int k = it.b, last = it.d - 1;
        dst = sW + (it.a + k) * kTreeT + b;
        m = x[k * kTreeT] * sDi[k * kTreeT + b];
        for (int p = part; p <= last; p += 4 * parts) {
          S u[4], v[4], d[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const TAnc q = treeAnc(g, tb, it.c + (p + t * parts <= last ? p + t * parts : last));
            u[t] = x[q.a * kTreeT];
            v[t] = sW[(q.rp + k) * kTreeT + b];
            d[t] = sDi[q.a * kTreeT + b];
            d[t] = p + t * parts <= last ? d[t] : S(0);
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) acc += u[t] * (v[t] * d[t]);
        }
      }
      acc = treePartSum(acc, sh);
      if (on && part == 0) {
        *dst = fac ? m - acc : -(m + acc);
        if (fac && it.a == it.b) sDi[it.c * kTreeT + b] = S(1) / (m - acc);
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
         ((state > w ? state : w) + (size_t)(g.nnz + 2 * g.nv) * kTreeT) * sizeof(S);
}
template<class S>
__device__ __forceinline__ TreeRow<S> treeMinvEntry(const TProg& g, const int16_t* tb, const S* sW, const S* sDi, int e) {
  const int c = __umulhi(e, g.nvMagic), r = e - c * g.nv;
  const int lo = r < c ? r : c, hi = r < c ? c : r;
  const int n = reinterpret_cast<const uint8_t*>(tb + g.oCommon)[e], cl = tb[g.oCp + lo];
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
  S* sM = reinterpret_cast<S*>(tb + ((g.nTabFactor + 7) & ~7));
  S* sDi = sM + (g.nnz + g.nv) * kTreeT;
  S* sW = sDi + g.nv * kTreeT;
  treeMassTile<S>(g, tb, g.nTabFactor, mc, gq, b0, nb, sW, sM);
  treeFactor<S>(g, tb, sM, sDi, sW);
  for (int e = threadIdx.x; e < g.nv * g.nv; e += blockDim.x) treePut(gX, e, treeMinvEntry<S>(g, tb, sW, sDi, e), b0, nb);
}

}  // namespace rbd
