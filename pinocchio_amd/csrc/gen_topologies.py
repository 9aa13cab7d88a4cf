"""Build step: emit the compile-time topologies the kernels are instantiated for.

For every bundled model family (pinocchio_amd.models) this writes, under csrc/_gen/:
  topologies.inc          one `struct Topo_<name>` per topology (parents, joint types and
                          the derived TopoData, see topo.hpp)
  inst_<name>_<fam>.hip   the kernel instantiations of one kernel family for that topology
                          (separate units so that they compile in parallel)
  ops_<name>.cpp          the launcher table of the topology, assembled from its families
  registry.inc            the list of launcher tables the runtime searches at model upload
  units.mk                the list of generated units for the Makefile

Only the topology (parents and joint types) is baked in; placements, inertias, armature
and gravity are run-time constants, so any model with one of these trees runs on the
prebuilt kernels.

A user's robots join the list at build time: `make -C pinocchio_amd/csrc
ROBOTS=a.urdf,b.xml:freeflyer` (URDF or MJCF files; `:freeflyer` for a floating base) adds
each file's tree under the name robot_<file stem>[_ff], unless an identical tree is listed
already; trees not in depth-first order get the RNEA / ABA / kinematics families only.
"""
from __future__ import annotations

import argparse
import os
import re
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(os.path.dirname(HERE)))

from pinocchio_amd import models as M  # noqa: E402

# multi-wave variants of a family's kernels: (kernel, scalar, parameter list, wave counts)
_VEC3 = "const {s}*, int64_t, CView<{s}>, CView<{s}>, CView<{s}>, View<{s}>"
_RNEAD = ("const float*, int64_t, CView<float>, CView<float>, CView<float>, View<float>, View<float>, "
          "View<float>, int")
WAVE_KERNELS = {
    "dyn": [("k_aba_waves", "float", _VEC3.format(s="float"), (2, 4)),
            ("k_aba_waves", "double", _VEC3.format(s="double"), (4,)),
            ("k_rnea_waves", "float", _VEC3.format(s="float"), (4,)),
            ("k_rnea_waves", "double", _VEC3.format(s="double"), (4,))],
    "rnead": [("k_rnead", "float", _RNEAD, (4,))],
    "crba": [("k_crba_waves", s, f"const {s}*, int64_t, CView<{s}>, View<{s}>, int", (4,)) for s in ("float", "double")],
    "chol": [("k_chol_waves", f"{i}, {c}", f"int64_t, CView<{i}>, View<{c}>, View<{c}>", (4,))
             for i, c in (("float", "double"), ("double", "double"), ("float", "float"))],
}
# unit name suffix per scalar (or input and factor scalar)
SCALAR_TAG = {"float": "", "double": "d", "float, double": "fd", "double, double": "dd", "float, float": "ff"}
WAVE_TAG = {"k_rnea_waves": "rnea_"}  # units of a family's second multi-wave kernel
WAVE_COND = {"k_aba_waves": "abaSplitPaysFor<Topo_{name}, {sc}, {g}>()",
             "k_rnea_waves": "rneaSplitPaysFor<Topo_{name}, {sc}, {g}>()",
             "k_crba_waves": "crbaSplitPaysFor<Topo_{name}, {sc}, {g}>()",
             "k_chol_waves": "cholSplitPaysFor<Topo_{name}, {sc}, {g}>()",
             "k_rnead": "rneadSplitPays<Topo_{name}, {g}>()"}

DYN = ["dyn", "kin"]
FULL = ["dyn", "kin", "crba", "chol", "rnead", "abads", "kkt"]

# Tree of pinocchio's sample URDF robot models/simple_humanoid.urdf read with a free-flyer
# root (pinocchio_amd/urdf.py; 29 revolute joints, nq 36, nv 35): parents and joint
# types only -- its inertias and placements are run-time data like every model's.
SIMPLE_HUMANOID_PARENTS = [0, 0, 1, 2, 3, 4, 5, 6, 1, 8, 9, 10, 11, 12, 1, 14, 15, 16, 17, 18, 19, 20, 21, 22, 16, 24,
                           25, 26, 27, 28, 29]
SIMPLE_HUMANOID_TYPES = [0, 1, 2, 3, 4, 3, 3, 2, 2, 3, 4, 3, 3, 2, 3, 2, 4, 3, 2, 4, 3, 4, 3, 2, 3, 2, 4, 3, 4, 3, 2]


def simple_humanoid_topology():
    n = len(SIMPLE_HUMANOID_PARENTS)
    return M.ModelDesc("simple_humanoid", SIMPLE_HUMANOID_PARENTS, SIMPLE_HUMANOID_TYPES,
                       M.np.tile(M.np.concatenate([M.np.eye(3).ravel(), M.np.zeros(3)]), (n, 1)),
                       M.np.tile([1.0, 0, 0, 0, 0.1, 0, 0.1, 0, 0, 0.1], (n, 1)))


# (name, builder, kernel families to instantiate)
TOPOLOGIES = [
    ("simple_humanoid", simple_humanoid_topology, FULL),
    ("manipulator6", M.manipulator6, FULL),
    ("arm7", M.arm7, FULL),
    ("quadruped18", M.quadruped18, FULL),
    ("humanoid36", M.humanoid36, FULL),
    ("random60", M.random60, DYN),
    ("pendulum", M.pendulum, FULL),
    ("free_body", M.free_body, FULL),
]


# compiled mixes for the one-launch mixed-robot kernel: (name, topologies)
MIXES = [
    ("bench4", ["arm7", "quadruped18", "humanoid36", "random60"]),
]


def mix_unit(name, topos):
    decl = "".join(f"const TopoOps* ops_{t}();\n" for t in topos)
    tlist = ", ".join(f"Topo_{t}" for t in topos)
    ops = ", ".join(f"ops_{t}()" for t in topos)
    return ("// generated by gen_topologies.py -- do not edit\n#include \"../instantiate.hpp\"\nnamespace rbd {\n"
            + decl +
            f"static void launch_mix_{name}(hipStream_t st, unsigned grid, const MultiGroup* g, const MultiTile* t) {{\n"
            f"  hipLaunchKernelGGL((k_multi<{tlist}>), dim3(grid), dim3(kTile), 0, st, g, t);\n}}\n"
            f"const MixOps* mix_{name}() {{\n"
            f"  static const MixOps m = {{\"{name}\", {len(topos)}, {{{ops}}}, &launch_mix_{name}}};\n"
            "  return &m;\n}\n}  // namespace rbd\n")


def topo_struct(name, m):
    nj = m.njoints
    par = ", ".join(str(int(x)) for x in m.parents)
    typ = ", ".join(str(int(x)) for x in m.jtype)
    return (f"struct Topo_{name} {{\n"
            f"  static constexpr int NJ = {nj};\n"
            f"  static constexpr int parent[NJ] = {{{par}}};\n"
            f"  static constexpr int type[NJ] = {{{typ}}};\n"
            f"  static constexpr TopoData<NJ> T = makeTopo<NJ>(parent, type);\n"
            f"  static constexpr const char* name = \"{name}\";\n"
            f"}};\n")


def depth_first(parents):
    """True when every joint's subtree is the index range right after it (crba.hxx's
    compact, depth-first numbering): joint i's parent is joint i - 1 or one of its ancestors"""
    for i in range(2, len(parents)):
        a = i - 1
        while a > 0 and a != parents[i]:
            a = parents[a]
        if a != parents[i]:
            return False
    return True


def robot_topologies(spec, known):
    """extra (name, builder, families) entries for ROBOTS=path[:freeflyer],..."""
    from pinocchio_amd import mjcf, urdf
    out = []
    seen = {(tuple(int(x) for x in m.parents), tuple(int(x) for x in m.jtype)) for m in known}
    for item in filter(None, (x.strip() for x in spec.split(","))):
        path, _, root = item.partition(":")
        root = root or "fixed"
        if root not in ("fixed", "freeflyer"):
            raise ValueError(f"{item}: the root is 'fixed' or 'freeflyer'")
        parse = mjcf.parse if path.lower().endswith(".xml") else urdf.parse
        desc = parse(path, root=root)
        key = (tuple(int(x) for x in desc.parents), tuple(int(x) for x in desc.jtype))
        if key in seen:
            continue
        seen.add(key)
        stem = re.sub(r"[^A-Za-z0-9_]", "_", os.path.splitext(os.path.basename(path))[0])
        name = f"robot_{stem}" + ("_ff" if root == "freeflyer" else "")
        out.append((name, lambda d=desc: d, FULL if depth_first(desc.parents) else DYN))
    return out


def main(out_dir=None, robots=""):
    out_dir = out_dir or os.path.join(HERE, "_gen")
    os.makedirs(out_dir, exist_ok=True)
    topologies = list(TOPOLOGIES)
    if robots:
        topologies += robot_topologies(robots, [fn() for _, fn, _ in TOPOLOGIES])
    parts = ["// generated by gen_topologies.py -- do not edit\n#pragma once\n#include \"../topo.hpp\"\n"
             "namespace rbd {\n"]
    for name, fn, _ in topologies:
        parts.append(topo_struct(name, fn()))
    parts.append("}  // namespace rbd\n")
    _write(os.path.join(out_dir, "topologies.inc"), "".join(parts))
    reg = ["// generated by gen_topologies.py -- do not edit\n"]
    units = []
    for name, _, fams in topologies:
        for fam in fams:
            # the multi-wave kernel variants compile in units of their own (explicit
            # instantiation there, extern declaration here) so the build parallelises
            ext = "".join(f"extern template __global__ void {k}<Topo_{name}, {sc}, {g}>({sig});\n"
                          for k, sc, sig, gs in WAVE_KERNELS.get(fam, []) for g in gs)
            _write(os.path.join(out_dir, f"inst_{name}_{fam}.hip"),
                   "// generated by gen_topologies.py -- do not edit\n"
                   f"#include \"../instantiate.hpp\"\nnamespace rbd {{\n{ext}}}\nRBD_FILL({name}, {fam})\n")
            units.append(f"inst_{name}_{fam}")
            for k, sc, sig, gs in WAVE_KERNELS.get(fam, []):
                for g in gs:
                    cond = WAVE_COND[k].format(name=name, g=g, sc=sc)
                    tag = f"{WAVE_TAG.get(k, '')}w{g}" + SCALAR_TAG[sc]
                    _write(os.path.join(out_dir, f"inst_{name}_{fam}_{tag}.hip"),
                           "// generated by gen_topologies.py -- do not edit\n"
                           "#include \"../instantiate.hpp\"\nnamespace rbd {\n"
                           f"void* keep_{k}_{name}_{tag}() {{\n"
                           f"  if constexpr ({cond}) return (void*)&{k}<Topo_{name}, {sc}, {g}>;\n"
                           "  else return nullptr;\n}\n}  // namespace rbd\n")
                    units.append(f"inst_{name}_{fam}_{tag}")
        decl = "".join(f"void fill_{name}_{fam}(TopoOps&);\n" for fam in fams)
        calls = "".join(f"      fill_{name}_{fam}(o);\n" for fam in fams)
        _write(os.path.join(out_dir, f"ops_{name}.hip"),
               "// generated by gen_topologies.py -- do not edit\n"
               "#include \"../ops.hpp\"\n#include \"../kernels_common.hpp\"\n#include \"topologies.inc\"\n"
               "namespace rbd {\n" + decl +
               "template<class TP> TopoOps opsBase() {\n  TopoOps o{};\n  o.name = TP::name;\n"
               "  o.njoints = TP::NJ;\n  o.parent = TP::parent;\n  o.type = TP::type;\n  o.nq = TP::T.nq;\n"
               "  o.nv = TP::T.nv;\n  o.compact = TP::T.compact ? 1 : 0;\n  return o;\n}\n"
               f"const TopoOps* ops_{name}() {{\n  static const TopoOps ops = [] {{\n"
               f"      TopoOps o = opsBase<Topo_{name}>();\n" + calls +
               "      return o;\n  }();\n  return &ops;\n}\n}  // namespace rbd\n")
        units.append(f"ops_{name}")
        reg.append(f"RBD_REGISTER({name})\n")
    mixreg = ["// generated by gen_topologies.py -- do not edit\n"]
    for name, topos in MIXES:
        _write(os.path.join(out_dir, f"mix_{name}.hip"), mix_unit(name, topos))
        units.append(f"mix_{name}")
        mixreg.append(f"RBD_REGISTER_MIX({name})\n")
    _write(os.path.join(out_dir, "mixes.inc"), "".join(mixreg))
    _write(os.path.join(out_dir, "registry.inc"), "".join(reg))
    _write(os.path.join(out_dir, "units.mk"), "UNITS := " + " ".join(units) + "\n")
    return units


def _write(path, text):
    if os.path.exists(path) and open(path).read() == text:
        return
    with open(path, "w") as f:
        f.write(text)


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("out_dir", nargs="?", default=None)
    ap.add_argument("--robots", default="", help="URDF / MJCF files, comma separated, each optionally :freeflyer")
    a = ap.parse_args()
    main(a.out_dir or None, a.robots)
