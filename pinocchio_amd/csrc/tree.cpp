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
      g.nvlev = std::max(g.nvlev, dl[c] + 1);
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
  // items by dof level (8-byte records): column entries of the factorisation, then W
  std::vector<int> lvl, items;
  for (int l = 0; l < g.nvlev; ++l) {
    lvl.push_back((int)items.size() / 4);
    for (int j = 0; j < nv; ++j)
      if (dl[j] == l) {
        items.insert(items.end(), {rp[j], rp[j], j, sub[j]});
        for (int r : anc[j]) items.insert(items.end(), {rp[r], rp[j], j, sub[j]});
      }
    lvl.push_back((int)items.size() / 4);
    for (int r = 0; r < nv; ++r)
      if (dl[r] == l)
        for (int k = r + 1; k < r + sub[r]; ++k)
          items.insert(items.end(), {rp[r], k, cp[k] + l + 1, dl[k] - 1 - l});
  }
  lvl.push_back((int)items.size() / 4);
  g.oLvl = flat(lvl);
  while (tab.size() & 3) tab.push_back(0);
  g.oItems = flat(items);
  // common strict ancestors of each pair of dofs
  std::vector<uint8_t> com((size_t)nv * nv + 1);
  for (int c = 0; c < nv; ++c)
    for (int r = 0; r < nv; ++r) {
      size_t k = 0;
      while (k < anc[r].size() && k < anc[c].size() && anc[r][k] == anc[c][k]) ++k;
      com[(size_t)c * nv + r] = (uint8_t)k;
    }
  g.oCommon = (int)tab.size();
  for (size_t k = 0; k + 1 < com.size(); k += 2) tab.push_back((int16_t)(com[k] | com[k + 1] << 8));
  g.nTabFactor = (int)tab.size();
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

namespace {

constexpr size_t kLdsMax = 160 * 1024;

// grid of treeTile(): a multiple of 8 covering the tiles
unsigned treeGrid(int64_t B) {
  const int64_t tiles = (B + kTreeT - 1) / kTreeT;
  return (unsigned)((tiles + 7) / 8 * 8);
}
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

// Measured on an MI355X, us per synchronous call, lane per configuration / tree-parallel.
// Trees without kernels of their own: faster at every size (27 joints, CRBA 232 / 22 at one
// configuration, 1009 / 52 at 16,384 by rows, 494 / 178 at 65,536 batch-fastest; Minv 884 /
// 42, 2118 / 155, 2749 / 513).
// Output by rows: 36 dofs 53 / 23 at one configuration, 1078 / 58 at 16,384, 4346 / 187 at
// 65,536 (Minv 103 / 49, 2144 / 202, 8778 / 704).  Matrices of a few hundred bytes stay
// where they were: one configuration is a few cache lines and the serial walk is short (6
// dofs: equal up to 16,384, FP64 21 / 28 there).
// Batch-fastest output: as long as the lane-per-configuration kernel has less than about
// one wave per SIMD to hide its serial walk (36 dofs CRBA 53 / 33 at 4,096, 53 / 46 at 8,192,
// 53 / 67 at 16,384; FP64 58 / 50 at 4,096, 58 / 82 at 8,192; Minv 105 / 65 at 4,096,
// 110 / 112 at 8,192).  FP64 Minv was one solve launch per column: 1627 / 352 at 16,384.
bool treePays(TreeOp op, bool prebuilt, bool rows, int nv, int es, int64_t B) {
  if (!prebuilt) return true;
  if (op == TreeOp::kMinv && es == 8) return true;
  if (rows) return nv * nv * es > 512;
  if (nv < 12) return false;
  return op == TreeOp::kCrba ? B * es <= 32768 : B <= 6144;
}

template<class S> bool treeCrba(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, View<S> M, int upper) {
  const TProg* g = prog(m);
  if (!g || B <= 0) return false;
  const size_t lds = treeCrbaLds<S>(*g);
  if (!allow(&t_crba<S>, lds)) return false;
  hipLaunchKernelGGL((t_crba<S>), dim3(treeGrid(B)), dim3(treeThreads(*g)), lds, st, *g, mc, B, q, M, upper);
  return true;
}

template<class S> bool treeMinv(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, View<S> X) {
  const TProg* g = prog(m);
  if (!g || B <= 0) return false;
  const size_t lds = treeMinvLds<S>(*g);
  if (!allow(&t_minv<S>, lds)) return false;
  hipLaunchKernelGGL((t_minv<S>), dim3(treeGrid(B)), dim3(treeThreads(*g)), lds, st, *g, mc, B, q, X);
  return true;
}

template bool treeCrba<float>(hipStream_t, GM, const float*, int64_t, CView<float>, View<float>, int);
template bool treeCrba<double>(hipStream_t, GM, const double*, int64_t, CView<double>, View<double>, int);
template bool treeMinv<float>(hipStream_t, GM, const float*, int64_t, CView<float>, View<float>);
template bool treeMinv<double>(hipStream_t, GM, const double*, int64_t, CView<double>, View<double>);

}  // namespace rbd
