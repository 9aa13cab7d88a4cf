"""The dispatch rules that choose between the tree-parallel kernels and the lane-per-configuration
ones: host functions of the library, no GPU.  Each row is a call whose two sides are given beside
the rule (tree.cpp), at sizes where they differ by more than the spread of the timings."""
import ctypes

import pytest

import pinocchio_amd as pa


class TreeShape(ctypes.Structure):
    _fields_ = [("joints", ctypes.c_int), ("nv", ctypes.c_int), ("nlev", ctypes.c_int)]


PENDULUM, FREE_BODY, CHAIN2, CHAIN5 = (1, 1, 1), (1, 6, 1), (2, 2, 2), (5, 5, 5)
CHAIN30, STAR4, HUMANOID = (30, 30, 30), (4, 4, 1), (31, 36, 10)


def rule(symbol, *args):
    fn = getattr(pa.lib(), symbol)
    fn.restype = ctypes.c_bool
    return fn(*args)


def dyn(aba, tree, es, B):
    return rule("_ZN3rbd11treeDynPaysEbNS_9TreeShapeEil", ctypes.c_bool(aba), TreeShape(*tree), ctypes.c_int(es),
                ctypes.c_int64(B))


@pytest.mark.parametrize("tree,aba,es,B,pays", [
    (PENDULUM, True, 4, 262144, False), (PENDULUM, False, 4, 65536, False), (FREE_BODY, True, 4, 65536, False),
    (FREE_BODY, True, 8, 16384, False), (CHAIN2, False, 4, 65536, False), (CHAIN2, True, 4, 65536, False),
    (CHAIN5, True, 4, 32768, False), (CHAIN5, False, 4, 65536, False), (STAR4, False, 4, 131072, False),
    (CHAIN5, True, 8, 8192, True), (STAR4, True, 4, 4096, True), (HUMANOID, False, 4, 16384, True),
    (HUMANOID, True, 4, 32768, True), (HUMANOID, True, 4, 65536, False), (CHAIN30, False, 4, 16384, False)])
def test_rnea_and_aba(tree, aba, es, B, pays):
    assert dyn(aba, tree, es, B) is pays
