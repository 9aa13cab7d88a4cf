// tree.cpp -- tables and launchers of the tree-parallel kernels (k_tree.hpp).
#include <algorithm>
#include <cstring>
#include <vector>

#include "generic.hpp"
#include "k_tree.hpp"
#include "runtime.hpp"
#include "tree.hpp"

namespace rbd {

// Tables of a tree whose numbering is depth first (a dof's subtree is the index range after
// it), appended to `words`; null for other trees and for patterns beyond the 16-bit entries.
// Part of every model's upload: the tables share the model's one buffer.
TreeProgram* buildTreeProgram(int nj, const int* parents, const int* types, std::vector<int32_t>& words) {
  std::vector<int> iq(nj, 0), iv(nj, 0), nvj(nj, 0), depth(nj, 0);
  int maxDepth = 0;
  TProg g{};
  g.nj = nj;
  for (int j = 1; j < nj; ++j) {
    int a = j - 1;  // depth first: the parent is j - 1 or one of its ancestors
    while (a > 0 && a != parents[j]) a = parents[a];
    if (a != parents[j]) return nullptr;
    const bool ff = types[j] == JT_FF;
    iq[j] = g.nq;
    iv[j] = g.nv;
    nvj[j] = ff ? 6 : 1;
    g.nq += ff ? 7 : 1;
    g.nv += nvj[j];
    depth[j] = parents[j] == 0 ? 1 : depth[parents[j]] + 1;
    maxDepth = std::max(maxDepth, depth[j]);
  }
  const int nv = g.nv;
  std::vector<int> dofJ(nv), dl(nv), cp(nv + 1, 0), sub(nv, 1), rp(nv), subJ(nj, 1);
  std::vector<std::vector<int>> anc(nv);
  for (int j = 1; j < nj; ++j) {
    for (int a = parents[j]; a > 0; a = parents[a]) subJ[a] += 1;
    for (int k = 0; k < nvj[j]; ++k) {
      const int c = iv[j] + k, p = parents[j];
      const int up = k > 0 ? c - 1 : (p > 0 ? iv[p] + nvj[p] - 1 : -1);
      if (up >= 0) {
        anc[c] = anc[up];
        anc[c].push_back(up);
      }
      dofJ[c] = j;
      dl[c] = (int)anc[c].size();
      cp[c + 1] = cp[c] + dl[c];
      for (int r : anc[c]) sub[r] += 1;
    }
  }
  g.nnz = cp[nv];
  if (nv < 1 || nv >= 256 || 2 * (g.nnz + nv) >= 32768 || nj * TJ_REC >= 32768) return nullptr;
  for (int r = 0, at = 0; r < nv; at += sub[r] - 1, ++r) rp[r] = at - (r + 1);
  g.nvMagic = (uint32_t)(((1ull << 32) + nv - 1) / nv);
  std::vector<int16_t> tab;
  tab.reserve(4096 + 12 * (size_t)g.nnz + (size_t)nv * nv / 2);
  auto flat = [&](const std::vector<int>& v) {
    const int o = (int)tab.size();
    tab.insert(tab.end(), v.begin(), v.end());
    return o;
  };
  for (int j = 0; j < nj; ++j) flat({parents[j], types[j], iq[j], iv[j], nvj[j]});
  // a list grouped by key 0 .. n - 1 of the joints: group starts, then the members
  auto grouped = [&](int n, auto key, int& oPtr, int& oList) {
    std::vector<int> ptr, list;
    for (int k = 0; k < n; ++k) {
      ptr.push_back((int)list.size());
      for (int j = 1; j < nj; ++j)
        if (key(j) == k) list.push_back(j);
    }
    ptr.push_back((int)list.size());
    oPtr = flat(ptr);
    oList = flat(list);
  };
  g.nlev = maxDepth;
  grouped(maxDepth, [&](int j) { return depth[j] - 1; }, g.oJLvl, g.oJList);
  grouped(nj, [&](int j) { return parents[j]; }, g.oKidP, g.oKid);
  g.nTabDyn = (int)tab.size();
  std::vector<int> up(parents, parents + nj);
  g.oJump = (int)tab.size();
  for (; (1 << g.nlog) < maxDepth; ++g.nlog) {
    flat(up);
    std::vector<int> next(nj, 0);
    for (int j = 1; j < nj; ++j) next[j] = up[up[j]];
    up = next;
  }
  g.oSubJ = flat(subJ);
  g.oDofJ = flat(dofJ);
  g.oDl = flat(dl);
  g.oRp = flat(rp);
  g.oSub = flat(sub);
  g.oCp = flat(cp);
  std::vector<int> pat;
  for (int c = 0; c < nv; ++c)
    for (int r : anc[c]) pat.insert(pat.end(), {r, rp[r]});
  while (tab.size() & 1) tab.push_back(0);
  g.oPat = flat(pat);
  g.nTab = (int)tab.size();
  // segments of treeFactor: a dof joins its predecessor's while that has no other child
  std::vector<int> nkid(nv, 0), seg, segOf(nv), slev;
  for (int c = 0; c < nv; ++c)
    if (!anc[c].empty()) nkid[anc[c].back()] += 1;
  for (int c = 0; c < nv; ++c) {
    const int p = anc[c].empty() ? -1 : anc[c].back();
    if (p >= 0 && p == c - 1 && nkid[p] == 1 && seg.back() < 4) {
      seg.back() += 1;
      segOf[c] = segOf[p];
    } else {
      segOf[c] = (int)seg.size() / 2;
      seg.insert(seg.end(), {c, 1});
      slev.push_back(p < 0 ? 0 : slev[segOf[p]] + 1);
      g.nslev = std::max(g.nslev, slev.back() + 1);
    }
  }
  // its items (8-byte records): phase 1 of a level with phase 3 of the level below, phase 2;
  // level -1 (only the last phase 3) first in the table of starts
  std::vector<int> lvl(4 * (g.nslev + 1)), items;
  for (int l = g.nslev - 1; l >= -1; --l) {
    int* at = &lvl[4 * (l + 1)];
    at[0] = (int)items.size() / 4;
    for (int s = 0; s < (int)slev.size(); ++s) {
      const int c0 = seg[2 * s], n = seg[2 * s + 1];
      if (slev[s] != l || sub[c0] == n) continue;  // nothing below: nothing to add
      for (int r : anc[c0]) items.insert(items.end(), {rp[r], r, s, -1});
      for (int i = 0; i < n; ++i) items.insert(items.end(), {rp[c0 + i], c0 + i, s, i});
    }
    at[1] = (int)items.size() / 4;
    for (int s = 0; s < (int)slev.size(); ++s) {
      const int c0 = seg[2 * s], n = seg[2 * s + 1];
      if (slev[s] != l + 1) continue;
      for (int k = c0 + n; k < c0 + sub[c0]; ++k)
        items.insert(items.end(), {k, s, cp[k] + dl[c0] + n, dl[k] - dl[c0] - n});
    }
    at[2] = (int)items.size() / 4;
    for (int s = 0; s < (int)slev.size(); ++s)
      if (slev[s] == l) {
        for (int r : anc[seg[2 * s]]) items.insert(items.end(), {rp[r], s, 0, 0});
        items.insert(items.end(), {0, s, 0, 1});
      }
    at[3] = (int)items.size() / 4;
  }
  g.oFSeg = flat(seg);
  g.oLvl = flat(lvl);
  while (tab.size() & 3) tab.push_back(0);
  g.oItems = flat(items);
  std::vector<int> segs;
  for (int c = 0; c < nv;) {
    int n = 1;
    while (n < 4 && c + n < nv && !anc[c + n].empty() && anc[c + n].back() == c + n - 1) ++n;
    segs.insert(segs.end(), {c, n});
    c += n;
  }
  g.oSeg = flat(segs);
  g.nseg = (int)segs.size() / 2;
  // common strict ancestors of each pair of dofs
  std::vector<uint8_t> com((size_t)nv * nv + 1);
  for (int c = 0; c < nv; ++c)
    for (int r = 0; r < nv; ++r) {
      size_t k = 0;
      while (k < anc[r].size() && k < anc[c].size() && anc[r][k] == anc[c][k]) ++k;
      com[(size_t)c * nv + r] = (uint8_t)k;
    }
  g.nTabFactor = (int)tab.size();
  g.oCommon = (int)tab.size();
  for (size_t k = 0; k + 1 < com.size(); k += 2) tab.push_back((int16_t)(com[k] | com[k + 1] << 8));
  g.oPairs = (int)tab.size();
  for (int c = 0; c < nv; ++c)
    for (int r = 0; r <= c; ++r) tab.push_back((int16_t)(r | c << 8));
  while (tab.size() & 3) tab.push_back(0);
  while (words.size() & 3) words.push_back(0);
  auto t = std::make_unique<TreeProgram>();
  t->word = words.size();
  t->g = std::make_unique<TProg>(g);
  words.resize(words.size() + tab.size() / 2);
  std::memcpy(words.data() + t->word, tab.data(), tab.size() * 2);
  return t.release();
}
void TreeProgram::place(const int32_t* dev) { g->tab = reinterpret_cast<const int16_t*>(dev + word); }

TreeProgram::TreeProgram() = default;
TreeProgram::~TreeProgram() = default;

bool gridFits(int64_t workgroups, int threads) { return workgroups < (int64_t(1) << 32) / threads; }

namespace {

constexpr size_t kLdsMax = 160 * 1024;

// grid of treeTile(): a multiple of 8 covering the tiles
int64_t treeTiles(int64_t B) { return ((B + kTreeT - 1) / kTreeT + 7) / 8 * 8; }
unsigned treeGrid(int64_t B) { return (unsigned)treeTiles(B); }
// dynamic LDS above the default 64 KB per workgroup needs the kernel attribute
template<class F> bool allow(F* fn, size_t bytes) {
  if (bytes <= 64 * 1024) return true;
  if (bytes > kLdsMax) return false;
  if (hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return true;
}
// threads per workgroup: two workers per dof, so that the columns of a matrix and the items
// of most levels are one round; a whole number of waves
unsigned treeThreads(const TProg& g) {
  const int t = (2 * g.nv * kTreeT + 63) / 64 * 64;
  return (unsigned)std::min(t, kTreeMaxThreads);
}
const TProg* prog(GM m) { return m->tree ? m->tree->g.get() : nullptr; }

}  // namespace

// Measured on an MI355X, us per synchronous call, lane per configuration / tree-parallel;
// FP32 unless said.
// Trees without kernels of their own: faster at every size from five dofs up (27 joints, CRBA
// 3996 / 130 at 65,536 by rows, 494 / 161 batch-fastest; Minv 7560 / 380, 2745 / 362; ABA
// derivatives 18223 / 1681, 7791 / 1721; chains of 5 to 40 joints and 12 joints at the root
// alike), but for
//  * the smallest trees, whose serial walk is a few us, beyond the batch that one round of
//    tiles covers.  CRBA: one joint 16 / 17 at 4,096, 16 / 21 at 65,536; a free flyer batch-
//    fastest 24 / 20 at 32,768, 24 / 26 at 65,536, FP64 25 / 21 at 16,384, 26 / 35 at 65,536; two
//    joints 18 / 18 at 16,384, 19 / 23 at 65,536; three 21 / 21 at 32,768, 31 / 34 at 131,072;
//    five batch-fastest 28 / 23 at 32,768, 29 / 32 at 65,536; four at the root FP64 26 / 23 at
//    32,768, 29 / 41 at 131,072, twelve 62 / 40, 74 / 99.  Minv: one joint 21 / 20 at 32,768,
//    22 / 30 at 131,072; a free flyer batch-fastest 52 / 42 at 65,536, 59 / 64 at 131,072 (FP64
//    266 / 195 at 262,144); four joints 38 / 33 at 65,536, four at the root 48 / 51 at 262,144.
//    Derivatives: one joint 28 / 32 at 4,096, 30 / 62 at 65,536; two 39 / 40 at 8,192, 40 / 56 at
//    32,768; three 101 / 103 at 65,536, 137 / 174 at 131,072; a free flyer batch-fastest 83 / 75 at
//    32,768, 117 / 117, 174 / 195 at 131,072; four at the root 54 / 50 at 32,768, 59 / 72 at 65,536.
//  * CRBA batch-fastest in FP64 beyond about 1 GiB of M (a tile writes 64 bytes of each row, the
//    rows a whole batch apart; not traced further): 31 joints 537 / 512 at 65,536,
//    973 / 1026 at 131,072, 1926 / 2415 at 262,144; 30 in a chain 1029 / 1028 at 131,072, 1995 /
//    2304; 18 dofs 593 / 580 at 262,144, 1108 / 1168 at 524,288.
// Trees with kernels of their own, output by rows: 36 dofs, CRBA 33 / 22 at one configuration,
// 1012 / 48 at 16,384, 4369 / 157 at 65,536 (Minv 71 / 41, 2048 / 124, 8867 / 441; ABA derivatives
// 211 / 87, 4967 / 371, 20686 / 1582).  Matrices of a few hundred bytes stay where they were, but
// for the derivatives: one configuration is a few cache lines and the serial walk is short (6
// dofs: equal up to 16,384, FP64 21 / 23 there; derivatives 60 / 56; of a single free flyer 42 /
// 42 at 8,192, 75 / 66 at 32,768; of a pendulum 25 / 29 at 1,024, 26 / 45 at 65,536).
// Batch-fastest output: where the lane-per-configuration kernels' walk is longer than the
// phases of the tiles of a CU (36 dofs, CRBA 33 / 22 at one configuration, 33 / 31 at 3,072,
// 33 / 37 at 5,120, FP64 36 / 30 at 1,024, 36 / 47 at 3,072; 18 dofs 21 / 21 at 2,048; Minv 75 /
// 59 at 6,144, 77 / 80 at 8,192; 18 dofs 34 / 32, 35 / 34, 36 / 46 at 12,288; derivatives 36 dofs
// 221 / 185 at 5,120, 225 / 205 at 8,192, 229 / 258 at 10,240, FP64 856 / 566 at 10,240, 926 / 973
// at 16,384; 18 dofs 75 / 71 at 5,120, 81 / 85 at 8,192, FP64 227 / 172 at 10,240, 235 / 254 at
// 16,384; 7 dofs 53 / 50 at 1,024, 53 / 52 at 4,096, FP64 73 / 57 at 4,096, 87 / 88 at 16,384).
// FP64 Minv is one solve launch per column there: 36 dofs 1611 / 298 at 16,384, 12213 / 4640 at
// 262,144; 7 dofs 91 / 85 at 65,536, 136 / 148 at 131,072; a pendulum 23 / 22 at 32,768, 23 / 28
// at 65,536.
bool treePays(TreeOp op, TreeShape t, bool prebuilt, bool rows, int es, int64_t B) {
  const int nv = t.nv;
  const int64_t n = B * es;
  if (!prebuilt) {
    switch (op) {
      case TreeOp::kCrba:
        if (nv < 3) return nv == 2 && n <= 65536;
        if (rows) return nv > 3 || n <= 131072;
        if (t.joints < 3 || nv < 6 || t.nlev < 2) return n <= 131072;
        return es == 4 || B * nv * nv <= int64_t(1) << 27;
      case TreeOp::kMinv:
        if (nv < 3) return n <= 131072;
        return rows || es == 8 || (t.joints > 1 && nv > 4) || n <= 262144;
      case TreeOp::kDeriv:
        if (nv < 4) return nv == 3 ? n <= 262144 : nv == 2 && n <= 32768;
        return rows || t.nlev > 1 || t.joints > 7 || n <= 131072;
    }
  }
  if (op == TreeOp::kDeriv) {
    if (t.joints < 2) return rows && nv > 1 && n > 65536;
    return rows || B * 4 <= (nv < 12 ? 2048 : 5120) * es;
  }
  if (op == TreeOp::kMinv && es == 8) return (nv > 1 && rows) || nv >= 12 || n <= (nv > 1 ? 524288 : 262144);
  if (rows) return nv * nv * es > 512;
  if (nv < 12) return false;
  return op == TreeOp::kCrba ? n <= 12288 : B <= 6144;
}

// The tree-parallel sweeps take a few phases per level with most lanes idle.  While all
// tiles are resident (some 16,384 FP32 configurations) a call takes one tile's time; beyond,
// time grows with the batch, and the lane-per-configuration kernels win once they fill the
// chip: later for a shallow tree (a shorter sweep) and for one of many joints (a longer walk),
// at once for one or two joints.  us per call, lane per configuration / tree-parallel:
//   RNEA, 10 levels (31 joints) 76 / 32 at 1,024, 76 / 54 at 16,384, 79 / 73 at 24,576, 79 / 92
//   at 32,768; 10 in a chain 34 / 32, 35 / 36 (24,576), FP64 45 / 33 at 8,192, 46 / 51 at 16,384;
//   40 in a chain 108 / 72 at 4,096, 111 / 129 at 8,192; six 26 / 26 at 16,384, 26 / 28 at 24,576,
//   FP64 30 / 29, 31 / 40; 12 at the root 32 / 25 at 32,768, 34 / 32 at 65,536, 34 / 39 at 98,304;
//   three in a chain 20 / 20 at 1,024, 20 / 24 at 32,768; two 18 / 19 at 1,024, 19 / 30 at 65,536.
//   ABA, 10 levels 235 / 46 at 1,024, 413 / 261 at 32,768, 447 / 383 at 49,152, 485 / 518 at
//   65,536; 40 in a chain 465 / 240 at 8,192, 468 / 350 at 12,288, 473 / 460 at 16,384; six 81 / 65
//   at 32,768, 88 / 85 at 49,152, 91 / 103; five 32 / 32 at 16,384, 33 / 56 at 32,768; three 25 / 26
//   at 16,384, FP64 38 / 27 at 8,192, 38 / 40 at 16,384; six at the root 30 / 30 at 49,152, FP64
//   35 / 32 at 32,768; two 21 / 21 at 1,024, 21 / 23 at 16,384; one 18 / 33 at 65,536.
bool treeDynPays(bool aba, TreeShape t, int es, int64_t B) {
  const int64_t n = B * es;
  if (t.joints < 3) return false;
  if (aba) return n <= (t.joints < 6 ? 65536 : 30000 * t.joints) && n * t.nlev <= 1400000;
  return n <= 10923 * t.joints && n * t.nlev <= 655360;
}

template<class S> bool treeCrba(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, View<S> M, int upper) {
  const TProg* g = prog(m);
  if (!g || B <= 0) return false;
  const size_t lds = treeCrbaLds<S>(*g);
  if (!gridFits(treeTiles(B), (int)treeThreads(*g)) || !allow(&t_crba<S>, lds)) return false;
  hipLaunchKernelGGL((t_crba<S>), dim3(treeGrid(B)), dim3(treeThreads(*g)), lds, st, *g, mc, B, q, M, upper);
  return true;
}

template<class S> bool treeMinv(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, View<S> X) {
  const TProg* g = prog(m);
  if (!g || B <= 0) return false;
  const size_t lds = treeMinvLds<S>(*g);
  if (!gridFits(treeTiles(B), (int)treeThreads(*g)) || !allow(&t_minv<S>, lds)) return false;
  hipLaunchKernelGGL((t_minv<S>), dim3(treeGrid(B)), dim3(treeThreads(*g)), lds, st, *g, mc, B, q, X);
  return true;
}

template<class S>
bool treeRnea(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> a, View<S> tau) {
  const TProg* g = prog(m);
  if (!g || B <= 0) return false;
  const size_t lds = treeDynLds<S>(*g, kTreeRneaJnt);
  if (!allow(&t_rnea<S>, lds)) return false;
  hipLaunchKernelGGL((t_rnea<S>), dim3(treeGrid(B)), dim3(kTreeDynThreads), lds, st, *g, mc, B, q, v, a, tau);
  return true;
}
template<class S>
bool treeAba(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> tau, View<S> ddq) {
  const TProg* g = prog(m);
  if (!g || B <= 0) return false;
  const size_t lds = treeDynLds<S>(*g, kTreeAbaJnt);
  if (!allow(&t_aba<S>, lds)) return false;
  hipLaunchKernelGGL((t_aba<S>), dim3(treeGrid(B)), dim3(kTreeDynThreads), lds, st, *g, mc, B, q, v, tau, ddq);
  return true;
}
template bool treeRnea<float>(hipStream_t, GM, const float*, int64_t, CView<float>, CView<float>, CView<float>,
                              View<float>);
template bool treeRnea<double>(hipStream_t, GM, const double*, int64_t, CView<double>, CView<double>, CView<double>,
                               View<double>);
template bool treeAba<float>(hipStream_t, GM, const float*, int64_t, CView<float>, CView<float>, CView<float>,
                             View<float>);
template bool treeAba<double>(hipStream_t, GM, const double*, int64_t, CView<double>, CView<double>, CView<double>,
                              View<double>);

namespace {
// segments per round of the solve: two workgroups per CU where that allows any
template<class S> int treeSolveRounds(const TProg& g) {
  int R = 3;
  while (R > 1 && treeSolveLds<S>(g, R) > kLdsMax / 2) --R;
  return R;
}
}  // namespace
template<class S> size_t treeDerivEntries(GM m) {
  const TProg* g = prog(m);
  if (!g || treeRneadLds<S>(*g) > kLdsMax || treeSolveLds<S>(*g, treeSolveRounds<S>(*g)) > kLdsMax) return 0;
  return (size_t)treeWsEntries(*g);
}
template size_t treeDerivEntries<float>(GM);
template size_t treeDerivEntries<double>(GM);

template<class S>
bool treeAbaDeriv(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> a, View<S> Xq,
                  View<S> Xv, View<S> Minv, S* ws) {
  const TProg* g = prog(m);
  if (!g || B <= 0) return false;
  const int R = treeSolveRounds<S>(*g);
  const size_t l1 = treeRneadLds<S>(*g), l2 = treeSolveLds<S>(*g, R);
  if (!allow(&t_rnead<S>, l1) || !allow(&t_dsolve<S>, l2)) return false;
  const unsigned grid = treeGrid(B);
  // Three workgroups per tile while they find places of their own: two per CU, or one where the
  // solve takes more than half of the LDS (us per call, one / three: 36 dofs 98 / 88 at one
  // configuration, 104 / 97 at 1,344, 109 / 113 at 1,408; FP64, one per CU, 133 / 113 at 512,
  // 145 / 128 at 768, 148 / 149 at 1,024, 150 / 171 at 1,344; 18 dofs FP64, two per CU, 66 / 62 at 1,344,
  // 66 / 69 at 1,408; 30 in a chain FP64 220 / 218 at 768, 227 / 239 at 1,024).
  const unsigned y = grid <= (l2 <= kLdsMax / 2 ? 168 : 96) ? 3 : 1;
  hipLaunchKernelGGL((t_rnead<S>), dim3(grid), dim3(treeThreads(*g)), l1, st, *g, mc, B, q, v, a, ws);
  hipLaunchKernelGGL((t_dsolve<S>), dim3(grid, y), dim3(treeThreads(*g)), l2, st, *g, B, (const S*)ws, Xq, Xv, Minv, R);
  return true;
}

template bool treeAbaDeriv<float>(hipStream_t, GM, const float*, int64_t, CView<float>, CView<float>, CView<float>,
                                  View<float>, View<float>, View<float>, float*);
template bool treeAbaDeriv<double>(hipStream_t, GM, const double*, int64_t, CView<double>, CView<double>,
                                   CView<double>, View<double>, View<double>, View<double>, double*);
template bool treeCrba<float>(hipStream_t, GM, const float*, int64_t, CView<float>, View<float>, int);
template bool treeCrba<double>(hipStream_t, GM, const double*, int64_t, CView<double>, View<double>, int);
template bool treeMinv<float>(hipStream_t, GM, const float*, int64_t, CView<float>, View<float>);
template bool treeMinv<double>(hipStream_t, GM, const double*, int64_t, CView<double>, View<double>);

}  // namespace rbd
