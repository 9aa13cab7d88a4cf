"""The dispatch rules that choose between two kernels for a call: host functions of the library, no
GPU.  Each row is a call whose two sides are given beside the rule (tree.cpp, cholops.cpp, generic.cpp), at sizes
where they differ by more than the spread of the timings."""
import ctypes

import pytest

import pinocchio_amd as pa


class TreeShape(ctypes.Structure):
    _fields_ = [("joints", ctypes.c_int), ("nv", ctypes.c_int), ("nlev", ctypes.c_int)]


PENDULUM, FREE_BODY, CHAIN2, CHAIN5 = (1, 1, 1), (1, 6, 1), (2, 2, 2), (5, 5, 5)
CHAIN30, STAR4, HUMANOID, ARM7 = (30, 30, 30), (4, 4, 1), (31, 36, 10), (7, 7, 7)
CRBA, MINV, DERIV = range(3)


def rule(symbol, *args):
    fn = getattr(pa.lib(), symbol)
    fn.restype = ctypes.c_bool
    return fn(*args)


def dyn(aba, tree, es, B):
    return rule("_ZN3rbd11treeDynPaysEbNS_9TreeShapeEil", ctypes.c_bool(aba), TreeShape(*tree), ctypes.c_int(es),
                ctypes.c_int64(B))


def pays(op, tree, prebuilt, rows, es, B):
    return rule("_ZN3rbd8treePaysENS_6TreeOpENS_9TreeShapeEbbil", ctypes.c_int(op), TreeShape(*tree),
                ctypes.c_bool(prebuilt), ctypes.c_bool(rows), ctypes.c_int(es), ctypes.c_int64(B))


@pytest.mark.parametrize("tree,aba,es,B,expect", [
    (PENDULUM, True, 4, 262144, False), (PENDULUM, False, 4, 65536, False), (FREE_BODY, True, 4, 65536, False),
    (FREE_BODY, True, 8, 16384, False), (CHAIN2, False, 4, 65536, False), (CHAIN2, True, 4, 65536, False),
    (CHAIN5, True, 4, 32768, False), (CHAIN5, False, 4, 65536, False), (STAR4, False, 4, 131072, False),
    (CHAIN5, True, 8, 8192, True), (STAR4, True, 4, 4096, True), (HUMANOID, False, 4, 16384, True),
    (HUMANOID, True, 4, 32768, True), (HUMANOID, True, 4, 65536, False), (CHAIN30, False, 4, 16384, False)])
def test_rnea_and_aba(tree, aba, es, B, expect):
    assert dyn(aba, tree, es, B) is expect


@pytest.mark.parametrize("op,tree,rows,es,B,expect", [
    (CRBA, PENDULUM, True, 8, 262144, False), (CRBA, PENDULUM, False, 4, 65536, False),
    (CRBA, FREE_BODY, False, 8, 65536, False), (CRBA, CHAIN2, False, 4, 262144, False),
    (CRBA, HUMANOID, False, 8, 262144, False), (CRBA, CHAIN30, False, 8, 262144, False),
    (CRBA, FREE_BODY, True, 4, 262144, True), (CRBA, HUMANOID, False, 4, 262144, True),
    (CRBA, HUMANOID, True, 8, 262144, True), (CRBA, CHAIN30, False, 4, 262144, True),
    (MINV, PENDULUM, True, 8, 262144, False), (MINV, FREE_BODY, False, 4, 131072, False),
    (MINV, FREE_BODY, False, 8, 262144, True), (MINV, CHAIN30, False, 8, 262144, True),
    (DERIV, PENDULUM, True, 4, 16384, False), (DERIV, CHAIN2, True, 8, 65536, False),
    (DERIV, FREE_BODY, False, 8, 65536, False), (DERIV, STAR4, False, 4, 65536, False),
    (DERIV, CHAIN5, False, 4, 65536, True), (DERIV, HUMANOID, False, 8, 262144, True)])
def test_matrices_of_trees_without_kernels_of_their_own(op, tree, rows, es, B, expect):
    assert pays(op, tree, False, rows, es, B) is expect


@pytest.mark.parametrize("op,tree,rows,es,B,expect", [
    (MINV, ARM7, False, 8, 262144, False), (MINV, FREE_BODY, False, 8, 262144, False),
    (MINV, PENDULUM, True, 8, 262144, False), (MINV, ARM7, True, 8, 262144, True),
    (MINV, HUMANOID, False, 8, 262144, True), (DERIV, PENDULUM, True, 4, 65536, False),
    (DERIV, FREE_BODY, False, 4, 1024, False), (DERIV, FREE_BODY, True, 4, 65536, True),
    (DERIV, HUMANOID, False, 4, 4096, True), (DERIV, HUMANOID, False, 4, 16384, False),
    (CRBA, HUMANOID, True, 4, 1, True), (CRBA, HUMANOID, False, 4, 8192, False), (CRBA, ARM7, True, 4, 4096, False)])
def test_matrices_of_prebuilt_trees(op, tree, rows, es, B, expect):
    assert pays(op, tree, True, rows, es, B) is expect


@pytest.mark.parametrize("nv,rows,B,expect", [
    (36, True, 1, True), (36, True, 1024, True), (36, True, 4096, False), (36, True, 16384, False),
    (18, True, 1024, True), (18, True, 8192, False), (36, False, 16384, True), (36, False, 16385, False)])
def test_tree_factor_on_four_waves(nv, rows, B, expect):
    assert rule("_ZN3rbd15cholSplitPaysAtEibl", ctypes.c_int(nv), ctypes.c_bool(rows), ctypes.c_int64(B)) is expect


@pytest.mark.parametrize("only_j,es,B,expect", [
    (True, 8, 64, False), (True, 8, 4096, False), (True, 8, 16384, True), (True, 4, 64, True), (False, 8, 64, True)])
def test_kinematics_rows_of_run_time_topologies(only_j, es, B, expect):
    assert rule("_ZN3rbd10kinRunsPayEbil", ctypes.c_bool(only_j), ctypes.c_int(es), ctypes.c_int64(B)) is expect


@pytest.mark.parametrize("batch,per_tile,threads,fits", [
    (1 << 28, 8, 128, False),          # 6 dofs, tree-parallel: two threads per dof and configuration
    ((1 << 28) - 4096, 8, 128, True), (1 << 30, 64, 256, False),  # four waves per 64 configurations
    ((1 << 30) - 4096, 64, 256, True), (1 << 31, 64, 64, True)])
def test_batches_beyond_one_launch(batch, per_tile, threads, fits):
    """A launch of 2^32 threads and more is refused; a call of that size takes the kernel with fewer
    threads per configuration."""
    tiles = -(-batch // per_tile)
    assert rule("_ZN3rbd8gridFitsEli", ctypes.c_int64(tiles), ctypes.c_int(threads)) is fits
