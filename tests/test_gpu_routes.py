"""Kernels that serve a call only beyond (or only below) a size, against the FP64 oracle just past
each switch and with a ragged last tile: the lane-per-configuration CRBA, factor and ABA
derivatives of prebuilt trees, and those of run-time topologies whose tree-parallel state does
not fit the LDS.  Every 97th configuration and the last 70 are checked.

Bars (per configuration, infinity norm, relative) as the other tests of the same quantities: M
1e-5 in FP32 and 1e-12 in FP64, ABA derivatives 1e-4 and 1e-9, tau 1e-5, the FP64 factor 1e-9."""
import numpy as np
import pytest

import oracle
import pinocchio_amd as pa
from helpers import f32_round, inputs, rel_err_cols, rel_err_mats
from pinocchio_amd import models as M

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

F32, F64 = torch.float32, torch.float64


def _case(d, B, dt):
    x = inputs(d, B, k=41)
    x = f32_round(*x) if dt == F32 else x
    idx = np.unique(np.r_[np.arange(0, B, 97), np.arange(max(0, B - 70), B)])
    return x, tuple(y[:, idx] for y in x), idx


def _dev(x, layout, dt):
    return torch.tensor(np.ascontiguousarray(x.T if layout == "col" else x), dtype=dt, device="cuda")


def _mats(t, layout, nv, idx):
    return pa.Engine.mats_to_numpy(t[idx] if layout == "col" else t[:, idx].contiguous(), layout, nv)


@pytest.mark.parametrize("robot,dt,B", [
    ("quadruped18", F64, 10301), ("humanoid36", F64, 10301), ("arm7", F64, 4161), ("humanoid36", F32, 5185),
    ("humanoid36", F32, 16449), ("quadruped18", F32, 5185), ("arm7", F32, 2113), ("free_body", F64, 131),
    ("pendulum", F32, 131)])
def test_aba_derivatives_of_prebuilt_trees(gpu_ctx, robot, dt, B):
    d = getattr(M, robot)()
    e = pa.Engine(pa.Model(gpu_ctx, d), "batch")
    (q, v, _, tau), (sq, sv, _, st), idx = _case(d, B, dt)
    out = e.aba_derivatives(*(_dev(x, "batch", dt) for x in (q, v, tau)))
    for o, r in zip(out[:3], oracle.aba_derivatives(d, sq, sv, st)[:3]):
        assert rel_err_mats(_mats(o, "batch", d.nv, idx), r).max() < (1e-4 if dt == F32 else 1e-9)


@pytest.mark.parametrize("robot", ["humanoid36", "quadruped18"])
@pytest.mark.parametrize("dt,B", [(F32, 3137), (F32, 16321), (F32, 16449), (F64, 1601), (F64, 16449)])
def test_crba_of_prebuilt_trees(gpu_ctx, robot, dt, B):
    """Four waves by subtrees up to 16,384 configurations, two waves beyond: the whole matrix, and the
    upper triangle alone (a joint's own block is written whole, the rest of the lower triangle left)."""
    d = getattr(M, robot)()
    e = pa.Engine(pa.Model(gpu_ctx, d), "batch")
    (q, *_), (sq, *_), idx = _case(d, B, dt)
    Q, ref, nv = _dev(q, "batch", dt), oracle.crba(d, sq), d.nv
    bar = 1e-5 if dt == F32 else 1e-12
    assert rel_err_mats(_mats(e.crba(Q), "batch", nv, idx), ref).max() < bar
    out = e.crba(Q, out=torch.full((nv * nv, B), 7.0, dtype=dt, device="cuda"), upper_only=True)
    keep = np.triu(np.ones((nv, nv), dtype=bool))
    keep[:6, :6] = True
    got = _mats(out, "batch", nv, idx)
    assert rel_err_mats(np.where(keep, got, 0), np.where(keep, ref, 0)).max() < bar
    assert (got[:, ~keep] == 7.0).all()


@pytest.mark.parametrize("robot,layout,B", [
    ("humanoid36", "col", 1820), ("humanoid36", "col", 1821), ("quadruped18", "col", 3640), ("quadruped18", "col", 3649),
    ("humanoid36", "batch", 16383), ("humanoid36", "batch", 16385)])
@pytest.mark.parametrize("dt", [F32, F64])
def test_cholesky_of_prebuilt_trees(gpu_ctx, robot, layout, B, dt):
    """The FP64 factor on four waves and on one, of the same M (rounded to FP32 where it is given so)."""
    d = getattr(M, robot)()
    m = pa.Model(gpu_ctx, d)
    e = pa.Engine(m, layout)
    (q, *_), _, idx = _case(d, B, F64)
    Md = e.crba(_dev(q, layout, F64)).to(dt)
    U, D = e.cholesky_decompose(Md)
    Uo, Do, *_ = oracle.cholesky(d, _mats(Md.double(), layout, d.nv, idx), rhs=np.ones((d.nv, len(idx))))
    rows, cols = m.cholesky_pattern()
    pick = lambda t: (t[idx] if layout == "col" else t[:, idx].T).double().cpu().numpy()  # noqa: E731
    assert rel_err_cols(pick(D).T, Do.T).max() < 1e-9
    assert rel_err_cols(pick(U).T, Uo[:, rows, cols].T).max() < 1e-9


@pytest.mark.parametrize("robot", ["humanoid36", "random60"])
def test_rnea_wave_counts_agree(gpu_ctx, robot):
    """Inside a batch of 1,000 and one of 40,000 (beyond which the 60-dof tree runs one wave per tile)."""
    d = getattr(M, robot)()
    e = pa.Engine(pa.Model(gpu_ctx, d), "batch")
    (q, v, a, _), (sq, sv, sa, _), idx = _case(d, 40001, F32)
    ref = oracle.rnea(d, sq, sv, sa)
    tau = e.rnea(*(_dev(x, "batch", F32) for x in (q, v, a)))
    assert rel_err_cols(tau[:, idx].double().cpu().numpy(), ref).max() < 1e-5
    small = e.rnea(*(_dev(np.ascontiguousarray(x[:, :1000]), "batch", F32) for x in (q, v, a)))
    assert ((small - tau[:, :1000]).abs().amax(0) <= 2e-6 * tau[:, :1000].abs().amax(0)).all()


@pytest.mark.parametrize("layout", ["col", "batch"])
@pytest.mark.parametrize("tree,B", [(lambda: M.random_tree(60, 5), 131), (M.free_body, 16449), (M.pendulum, 4161)])
def test_run_time_topologies_beyond_the_tree_parallel_kernels(gpu_ctx, tree, B, layout):
    """FP64: 60 joints, whose state exceeds the LDS of a CU, and one joint at a batch where a lane per
    configuration is the faster."""
    d = tree()
    m = pa.Model(gpu_ctx, d, runtime_topology=True)
    e = pa.Engine(m, layout)
    (q, v, _, tau), (sq, sv, _, st), idx = _case(d, B, F64)
    Q, ref = _dev(q, layout, F64), oracle.crba(d, sq)
    up = np.triu(ref)
    if d.jtype[1] == M.JT_FREEFLYER:
        up[:, :6, :6] = ref[:, :6, :6]
    assert rel_err_mats(_mats(e.crba(Q), layout, d.nv, idx), ref).max() < 1e-12
    assert rel_err_mats(_mats(e.crba(Q, upper_only=True), layout, d.nv, idx), up).max() < 1e-12
    assert rel_err_mats(_mats(e.compute_minverse(Q), layout, d.nv, idx), np.linalg.inv(ref)).max() < 1e-9
    out = e.aba_derivatives(Q, *(_dev(x, layout, F64) for x in (v, tau)))
    for o, r in zip(out[:3], oracle.aba_derivatives(d, sq, sv, st)[:3]):
        assert rel_err_mats(_mats(o, layout, d.nv, idx), r).max() < 1e-9


def test_crba_beyond_a_tree_parallel_launch(gpu_ctx):
    """2^28 configurations by rows: 16 threads each would be a launch of 2^32, which the runtime refuses."""
    d = M.manipulator6()
    B, nv = 1 << 28, 6
    e = pa.Engine(pa.Model(gpu_ctx, d, runtime_topology=True), "col")
    gen = torch.Generator(device="cuda").manual_seed(5)
    q = torch.rand((B, d.nq), generator=gen, device="cuda") * 6.28 - 3.14
    out = e.crba(q)
    idx = np.r_[np.arange(70), np.arange(B // 2 - 5, B // 2 + 5), np.arange(B - 70, B)]
    ref = oracle.crba(d, np.ascontiguousarray(q[idx].double().cpu().numpy().T))
    assert rel_err_mats(_mats(out, "col", nv, idx), ref).max() < 1e-5


def test_aba_derivatives_beyond_the_lds_take_no_tree_workspace():
    """60 joints in FP64, whose packed path does not fit the LDS: the call allocates what the other path
    needs, the factor and ddq (43 MB here; the packed tiles would be 128 MiB)."""
    d, B = M.random_tree(60, 5), 8192
    c = pa.Context(0)
    m = pa.Model(c, d, runtime_topology=True)
    e = pa.Engine(m, "batch")
    x = [_dev(y, "batch", F64) for y in (lambda t: (t[0], t[1], t[3]))(inputs(d, B))]
    out = [torch.empty((d.nv * d.nv, B), dtype=F64, device="cuda") for _ in range(3)]
    ddq = torch.empty((d.nv, B), dtype=F64, device="cuda")
    e.aba_derivatives(*(y[:, :64].contiguous() for y in x))  # lane memory of the kernels, tables
    e.aba(*x, out=ddq)
    e.rnea_derivatives(x[0], x[1], x[2])
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    e.aba_derivatives(*x, out=out, ddq_out=ddq)
    nnz = len(m.cholesky_pattern()[0])
    assert free - torch.cuda.mem_get_info()[0] <= (nnz + 2 * d.nv) * B * 8 + (8 << 20)
