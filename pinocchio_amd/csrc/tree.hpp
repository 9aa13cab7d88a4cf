// tree.hpp -- launchers of the tree-parallel kernels (k_tree.hpp).  Host side; internal.
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <vector>

#include "ops.hpp"

namespace rbd {

struct TProg;

// Tables of one model's tree for the tree-parallel kernels: `word` is where they start in
// the model's table buffer, place() is told its device address.
struct TreeProgram {
  size_t word = 0;
  std::unique_ptr<TProg> g;
  void place(const int32_t* dev);
  TreeProgram();
  TreeProgram(const TreeProgram&) = delete;
  TreeProgram& operator=(const TreeProgram&) = delete;
  ~TreeProgram();
};
TreeProgram* buildTreeProgram(int nj, const int* parents, const int* types, std::vector<int32_t>& words);

struct TreeShape {
  int joints, nv, nlev;  // the universe not counted; levels of the tree
};
// Whether a call is faster on the tree-parallel kernels.  prebuilt: the tree has kernels of
// its own; rows: the output keeps a configuration's elements together (rs == 1); es: bytes
// of a scalar.
enum class TreeOp { kCrba, kMinv, kDeriv };
bool treePays(TreeOp op, TreeShape t, bool prebuilt, bool rows, int es, int64_t B);
// RNEA and ABA of a tree without kernels of its own
bool treeDynPays(bool aba, TreeShape t, int es, int64_t B);

// Each returns false, having launched nothing, when the model has no tree program, its state
// does not fit the LDS or the batch does not fit a launch: the caller then runs the
// lane-per-configuration kernels.
template<class S> bool treeCrba(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, View<S> M, int upper);
template<class S> bool treeMinv(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, View<S> X);
template<class S>
bool treeRnea(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> a, View<S> tau);
template<class S>
bool treeAba(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> tau, View<S> ddq);

// RNEA derivatives at a and the ABA-derivative solve; ws: treeDerivEntries<S>(m) scalars per
// configuration, the batch rounded up to a multiple of 8.  0: no tree program, or its state does
// not fit the LDS.
template<class S> size_t treeDerivEntries(GM m);
template<class S>
bool treeAbaDeriv(hipStream_t st, GM m, const S* mc, int64_t B, CView<S> q, CView<S> v, CView<S> a, View<S> Xq,
                  View<S> Xv, View<S> Minv, S* ws);

}  // namespace rbd
